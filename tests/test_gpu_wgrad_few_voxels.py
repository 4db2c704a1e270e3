"""Weight gradient of few voxels: the streaming kernel over one block, from one voxel to the last before the table streams by itself."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 5, 64, 65, 511])
@pytest.mark.parametrize("ci,co", [(8, 8), (16, 32), (72, 40), (128, 200), (512, 520)])
def test_against_float64(dtype, n, ci, co):
    g = torch.Generator().manual_seed(n + ci)
    flat = torch.randperm(10 ** 3, generator=g)[:n]
    coords = torch.stack([torch.zeros_like(flat), flat // 100, flat // 10 % 10, flat % 10], 1).int().cuda()
    cache = SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 10, 10, 10]), (3, 3, 3), (1, 1, 1), True)
    feats, grad = torch.randn(n, ci, generator=g).to(dtype).cuda(), torch.randn(n, co, generator=g).to(dtype).cuda()
    got, bias = nat.host().wgrad(grad, feats, cache, 27, True, 13)
    nmap = cache["neighbor_map"].view(torch.int32).cpu().long()
    f, gr = feats.cpu().double(), grad.cpu().double()
    u32, u16 = torch.finfo(torch.float32).eps, torch.finfo(dtype).eps
    for v in range(27):
        r = (nmap[:, v] >= 0).nonzero()[:, 0]
        want, size = gr[r].T @ f[nmap[r, v]], gr[r].abs().T @ f[nmap[r, v]].abs()
        # fp32 sums of at most n products, rounded once to the output type
        assert bool(((got[:, v].cpu().double() - want).abs() <= n * u32 * size + u16 * want.abs() + torch.finfo(dtype).tiny).all())
    assert bool(((bias.cpu().double() - gr.sum(0)).abs() <= n * u32 * gr.abs().sum(0) + u16 * gr.sum(0).abs() + torch.finfo(dtype).tiny).all())


def test_where_it_holds():
    tile = nat.lib().fgx_wgrad_short_tile
    assert tile(nat.DTYPE_CODE[torch.float32], nat.sz(100), 64, 64) == 0
    code = nat.DTYPE_CODE[torch.bfloat16]
    assert [tile(code, nat.sz(n), 64, 64) for n in (0, 1, 511, 512)] == [0, 64, 64, 0] and tile(code, nat.sz(9), 512, 512) == 128
