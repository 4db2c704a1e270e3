"""Bias gradient beside the weight gradient of narrow layers: ragged chunks, every channel count, values that are not finite."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction
from flexgemm_amd.ops.spconv import submanifold_conv3d as impl


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,ci,co", [(1, 8, 8), (127, 16, 24), (128, 32, 32), (129, 8, 32), (20000, 32, 16)])
@pytest.mark.parametrize("special", [False, True])
def test_bias_beside_narrow_weight_gradient(dtype, n, ci, co, special):
    g = torch.Generator().manual_seed(n + co)
    flat = torch.randperm(32 ** 3, generator=g)[:n]
    coords = torch.stack([torch.zeros_like(flat), flat // 1024, flat // 32 % 32, flat % 32], 1).int().cuda()
    cache = SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 32, 32, 32]), (3, 3, 3), (1, 1, 1), True)
    feats, grad = torch.randn(n, ci, generator=g).to(dtype).cuda(), (torch.randn(n, co, generator=g) + 0.5).to(dtype).cuda()
    if special:
        grad[n // 2, 1], grad[n // 3, 3] = float("inf"), float("nan")
    old = impl.spconv.NARROW_RESIDENT
    try:
        impl.spconv.NARROW_RESIDENT = "on"
        weight, bias = impl._wgrad(grad, feats, cache, 27, True, 13)
        alone = impl._wgrad(grad, feats, cache, 27)
        # a plan of before the last multiplier's entries were repeated in it
        header = cache["_narrow_plan_buf"][:256].view(torch.int32)
        assert int(header[1]) != 0
        header[1] = 0
        table = cache["_narrow_plan_buf"][256:256 + 128 * 64].view(torch.int16).view(128, 32)
        table[:, 27:30] = 448 * 64
        kept, bias_kept = impl._wgrad(grad, feats, cache, 27, True, 13) if n <= 128 else (weight, bias)
    finally:
        impl.spconv.NARROW_RESIDENT = old
    bits = lambda t: t.view(torch.int16)
    assert torch.equal(bits(weight), bits(alone)) and torch.equal(bits(weight), bits(kept)) and torch.equal(bits(bias), bits(bias_kept))
    want, size = grad.double().sum(0), grad.double().abs().sum(0)
    fine = torch.isfinite(want)
    assert torch.equal(torch.isfinite(bias), fine) and torch.equal(torch.isnan(bias), torch.isnan(want))
    # fp32 sums of n values, rounded once to the output type
    bound = n * torch.finfo(torch.float32).eps * size + torch.finfo(dtype).eps * want.abs() + torch.finfo(dtype).tiny
    assert bool(((bias.double() - want).abs() <= bound)[fine].all())
