"""Bias gradient made beside the streaming weight gradient: written by the product itself (one voxel block), and by the first
workgroups of each of the three reductions (several)."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,ci,co,tile,block_rows", [
    (700, 64, 72, 64, 1024), (1, 128, 128, 128, 1024), (3000, 96, 40, 64, 512), (3000, 128, 264, 128, 512), (3000, 256, 64, 64, 320),
    (3000, 16, 32, 32, 1024), (3500, 64, 64, 64, 64)])
def test_bias_beside_weight_gradient(monkeypatch, dtype, n, ci, co, tile, block_rows):
    g = torch.Generator().manual_seed(n + ci)
    flat = torch.randperm(16 ** 3, generator=g)[:n]
    coords = torch.stack([torch.zeros_like(flat), flat // 256, flat // 16 % 16, flat % 16], 1).int().cuda()
    cache = SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 16, 16, 16]), (3, 3, 3), (1, 1, 1), True)
    feats, grad = torch.randn(n, ci, generator=g).to(dtype).cuda(), torch.randn(n, co, generator=g).to(dtype).cuda()
    real = nat.table_lookup

    def lookup(*a, **k):
        s = real(*a, **k)
        s.tile_rows = s.tile_cols = tile
        s.stream, s.block_rows = 1, block_rows
        return s
    monkeypatch.setattr(nat, "table_lookup", lookup)
    weight, bias = nat.host().wgrad(grad, feats, cache, 27, True, 13)
    alone, _ = nat.host().wgrad(grad, feats, cache, 27, False, 13)
    assert torch.equal(weight, alone)
    want, size = grad.double().sum(0), grad.double().abs().sum(0)
    # fp32 sums of n values, rounded once to the output type
    bound = n * torch.finfo(torch.float32).eps * size + torch.finfo(dtype).eps * want.abs() + torch.finfo(dtype).tiny
    assert bool(((bias.double() - want).abs() <= bound).all())
