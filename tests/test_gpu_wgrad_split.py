"""fp32 weight gradient over the even split: its two tiles, ragged items, fewer pairs than workgroups, channels past a tile's edge, one
voxel block and several."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction



def coords_of(n, side, seed):
    g = torch.Generator().manual_seed(seed)
    flat = torch.randperm(side ** 3, generator=g)[:n]
    return torch.stack([torch.zeros_like(flat), flat // side ** 2, flat // side % side, flat % side], 1).int().cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [64, 96])
@pytest.mark.parametrize("n,blocks", [(1, 1), (63, 1), (700, 1), (700, 5), (2100, 3)])
@pytest.mark.parametrize("ci,co", [(4, 8), (64, 64), (96, 96), (100, 36), (68, 196)])
def test_tiles_against_float64(monkeypatch, tile, n, blocks, ci, co):
    torch.manual_seed(n + ci)
    cache = SubMConv3dFunction._compute_neighbor_cache(coords_of(n, 16, n), torch.Size([1, ci, 16, 16, 16]), (3, 3, 3), (1, 1, 1), True)
    feats, grad = torch.randn(n, ci, device="cuda"), torch.randn(n, co, device="cuda")
    real = nat.table_lookup

    def lookup(*a, **k):
        s = real(*a, **k)
        s.tile_rows = s.tile_cols = tile
        s.stream, s.block_rows = 1, -(-n // blocks)
        return s
    monkeypatch.setattr(nat, "table_lookup", lookup)
    got, bias = nat.host().wgrad(grad, feats, cache, 27, True, 13)
    nmap = cache["neighbor_map"].view(torch.int32).cpu().long()
    f, g = feats.cpu().double(), grad.cpu().double()
    want, size = torch.zeros(co, 27, ci, dtype=torch.double), torch.zeros(co, 27, ci, dtype=torch.double)
    for v in range(27):
        r = (nmap[:, v] >= 0).nonzero()[:, 0]
        want[:, v] = g[r].T @ f[nmap[r, v]]
        size[:, v] = g[r].abs().T @ f[nmap[r, v]].abs()
    # a sum of k products, in any order, is within k units in the last place of the sum of their magnitudes
    u = torch.finfo(torch.float32).eps
    assert bool(((got.cpu().double() - want).abs() <= (n + 256) * u * size).all())
    # ... and these sums of a few hundred products are far closer than that on the whole
    assert float((got.cpu().double() - want).norm()) <= 16 * u * float(want.norm()) + 1e-30
    assert bool(((bias.cpu().double() - g.sum(0)).abs() <= n * u * g.abs().sum(0)).all())


@pytest.mark.parametrize("n,ci,co,tile", [(2048, 96, 96, 96), (2047, 96, 96, None), (4096, 64, 64, 64), (4095, 64, 64, None), (12288, 256, 256, 64),
                                           (12289, 256, 256, None), (300000, 192, 160, None), (1 << 22, 96, 96, 96), (41700, 32, 32, None)])
def test_rule(n, ci, co, tile):
    L, rows = nat.lib(), C.c_int(0)
    got = L.fgx_wgrad_split_tile(nat.sz(n), ci, co, C.byref(rows))
    assert got == (tile or 0)
    if tile is not None:
        assert -(-n // rows.value) <= 2
        assert L.fgx_conv_wgrad_split_scratch_bytes(nat.sz(n), nat.sz(n), C.c_uint32(n), 27, ci, co, tile, rows.value) > 0


def test_sizes_out_of_range():
    size = nat.lib().fgx_conv_wgrad_split_scratch_bytes
    ok = [nat.sz(5000), nat.sz(5000), C.c_uint32(50000), 27, 96, 96, 96, 2500]
    assert size(*ok) > 0
    for at, value in ((0, nat.sz(0)), (2, C.c_uint32(0xFFFFFFFF)), (3, 0), (4, 6), (6, 32), (7, 0), (7, 60)):       # (60: 84 blocks x 27)
        assert size(*[value if i == at else a for i, a in enumerate(ok)]) == 0
