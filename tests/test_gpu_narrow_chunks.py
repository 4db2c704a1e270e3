"""Narrow layers of 3 x 3 x 3 kernels: row counts that give the workgroups no, one, two and more chunks of 128 rows, the last one full or of a row; chunks
with more distinct sources than slots."""
import numpy as np
import pytest
import torch

from flexgemm_amd.ops.spconv import SubMConv3dFunction, sparse_submanifold_conv3d, sparse_submanifold_conv3d_relu
from flexgemm_amd.ops.spconv import submanifold_conv3d as impl
from flexgemm_amd.workloads import reference_test_shell
from oracle import explicit_gemm as eg


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,ci,co", [(8 * 128, 32, 32), (256 * 128, 8, 16), (256 * 128 + 1, 16, 8), (512 * 128 - 127, 24, 24), (770 * 128, 8, 32),
                                     (1030 * 128 + 31, 32, 8), (1281 * 128 + 97, 16, 16)])
def test_narrow_layer_over_chunk_counts(gpu_device, dtype, n, ci, co):
    print(f"narrow layer n={n} {ci}->{co} {dtype}", flush=True)
    coords = torch.from_numpy(reference_test_shell(256)[:n]).to(gpu_device)
    assert len(coords) == n
    gen = torch.Generator().manual_seed(n)
    feats, grad = torch.randn(n, ci, generator=gen).to(dtype), torch.randn(n, co, generator=gen).to(dtype)
    weight, bias = (torch.randn(co, 27, ci, generator=gen) / (27 * ci) ** 0.5).to(dtype), torch.randn(co, generator=gen).to(dtype)
    f, g, w, b = (t.to(gpu_device) for t in (feats, grad, weight, bias))
    old = impl.spconv.NARROW_RESIDENT
    impl.spconv.NARROW_RESIDENT = "on"
    try:
        cache = SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 256, 256, 256]), (3, 3, 3), (1, 1, 1), True)
        out = impl._gather_gemm(f, w, b, cache, 0, False)
        gi = impl._gather_gemm(g, w, None, cache, 1, False)
        gw, gb = impl._wgrad(g, f, cache, 27, with_bias=True, bias_offset=13)
    finally:
        impl.spconv.NARROW_RESIDENT = old
    assert hasattr(cache, "_narrow_plan_buf") and cache["_narrow_overflows"] == 0
    nmap = cache.neighbor_map.cpu().view(torch.int32)
    ref = eg.forward(feats.double(), nmap, weight.view(co, 3, 3, 3, ci).double(), bias.double())
    ref_gi, ref_gw, ref_gb = eg.backward(grad.double(), feats.double(), nmap, weight.view(co, 3, 3, 3, ci).double())
    # one rounding to the type, and the fp32 roundings of a sum whose terms have random signs and a size of at most about one: it passes
    # through values of up to a few terms ** 0.5, and its terms' roundings of 2 ** -24 of them add up as the root once more
    half = torch.finfo(dtype).eps / 2
    for got, want, terms in ((out, ref, 27 * ci), (gi, ref_gi, 27 * co), (gw.view(co, 27, ci), ref_gw.view(co, 27, ci), n), (gb, ref_gb, n)):
        err = (got.cpu().double() - want).abs()
        assert bool((err <= half * want.abs() + torch.finfo(dtype).tiny + 4 * terms * 2.0 ** -24).all()), (tuple(want.shape), float(err.max()))


# A solid cube inside the shell, whose chunks overflow: the plan made beside the map sends every chunk's products to the kernel that reads the surplus
# from memory, and the weight gradient to the block-major kernel.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ci,co,dil,relu", [(32, 32, 1, False), (16, 24, 2, False), (24, 8, 2, True)])
def test_narrow_layer_with_overflowing_chunks(gpu_device, dtype, ci, co, dil, relu):
    res = 230
    side = np.arange(20, dtype=np.int32) + 38
    cube = np.stack(np.meshgrid(0, side, side, side, indexing="ij"), -1).reshape(-1, 4).astype(np.int32)
    coords = torch.from_numpy(np.concatenate([reference_test_shell(96), cube])).to(gpu_device)
    n = len(coords)
    print(f"narrow layer with overflowing chunks n={n} {ci}->{co} dilation={dil} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(ci)
    feats, grad = torch.randn(n, ci, generator=gen).to(dtype), torch.randn(n, co, generator=gen).to(dtype)
    weight, bias = (torch.randn(co, 3, 3, 3, ci, generator=gen) / (27 * ci) ** 0.5).to(dtype), torch.randn(co, generator=gen).to(dtype)
    f, w, b = (t.to(gpu_device).requires_grad_(True) for t in (feats, weight, bias))
    op = sparse_submanifold_conv3d_relu if relu else sparse_submanifold_conv3d
    out, cache = op(f, coords, torch.Size([1, ci, res, res, res]), w, b, None, (dil,) * 3)
    assert hasattr(cache, "_narrow_plan_buf")
    gi, gw, gb = torch.autograd.grad(out, (f, w, b), grad.to(gpu_device))
    assert cache["_narrow_overflows"] > 0
    nmap = cache.neighbor_map.cpu().view(torch.int32)
    ref = eg.forward(feats.double(), nmap, weight.double(), bias.double())
    if relu:
        grad = grad * (out.detach().cpu() > 0)
        ref = ref.clamp(min=0)
    ref_gi, ref_gw, ref_gb = eg.backward(grad.double(), feats.double(), nmap, weight.double())
    half = torch.finfo(dtype).eps / 2                       # (the bound: test_narrow_layer_over_chunk_counts)
    for got, want, terms in ((out, ref, 27 * ci), (gi, ref_gi, 27 * co), (gw.reshape(co, 27, ci), ref_gw.view(co, 27, ci), n), (gb, ref_gb, n)):
        err = (got.detach().cpu().double() - want).abs()
        assert bool((err <= half * want.abs() + torch.finfo(dtype).tiny + 4 * terms * 2.0 ** -24).all()), (tuple(want.shape), float(err.max()))
