"""Forward product of few voxels in one launch: ragged rows, columns and channel slabs, missing neighbors, bias, ReLU, and where the
operators take it."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import sparse_submanifold_conv3d, sparse_submanifold_conv3d_relu


def few(src, weight, bias, nmap, activation):
    n, v = nmap.shape
    guarded = torch.full((n * weight.shape[0] + 64,), 7.0, dtype=src.dtype, device="cuda")
    nat.check(nat.lib().fgx_conv_gemm_few(C.c_int(nat.DTYPE_CODE[src.dtype]), nat.ptr(src), nat.ptr(weight), nat.ptr(bias), nat.ptr(nmap), nat.sz(n),
                                          C.c_int(weight.shape[2]), C.c_int(weight.shape[0]), C.c_int(v), C.c_int(activation), nat.ptr(guarded), nat.stream()))
    assert bool((guarded[n * weight.shape[0]:] == 7).all())
    return guarded[:n * weight.shape[0]].view(n, weight.shape[0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000])
@pytest.mark.parametrize("ci,co,v", [(8, 1, 27), (32, 32, 27), (40, 30, 27), (64, 64, 27), (96, 65, 8), (128, 16, 27), (24, 130, 1), (256, 48, 32)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_against_float64(dtype, n, ci, co, v, with_bias):
    g = torch.Generator().manual_seed(n + ci + v)
    n_src = n + 3
    src = torch.randn(n_src, ci, generator=g).to(dtype)
    weight = (torch.randn(co, v, ci, generator=g) / (v * ci) ** 0.5).to(dtype)
    bias = torch.randn(co, generator=g).to(dtype) if with_bias else None
    nmap = torch.randint(0, n_src, (n, v), generator=g)
    nmap[torch.rand(n, v, generator=g) < 0.5] = -1
    rows = torch.where((nmap >= 0)[..., None], src.double()[nmap.clamp(min=0)], 0.0)
    want = torch.einsum("nvk,cvk->nc", rows, weight.double()) + (bias.double() if with_bias else 0)
    size = torch.einsum("nvk,cvk->nc", rows.abs(), weight.double().abs()) + (bias.double().abs() if with_bias else 0)
    dev = nmap.to(torch.int32).cuda()
    # fp32 sums of v * ci products, rounded once to the output type
    bound = (v * ci + 1) * torch.finfo(torch.float32).eps * size + torch.finfo(dtype).eps * want.abs() + torch.finfo(dtype).tiny
    for activation in (0, 1):
        ref = want.clamp(min=0) if activation else want
        got = few(src.cuda(), weight.cuda(), bias.cuda() if with_bias else None, dev, activation)
        assert bool(((got.cpu().double() - ref).abs() <= bound).all())
        assert torch.equal(got, few(src.cuda(), weight.cuda(), bias.cuda() if with_bias else None, dev, activation))


@pytest.mark.gpu
@pytest.mark.parametrize("n,ci,co", [(300, 32, 32), (300, 20, 24), (2000, 32, 48)])
def test_operators_take_it_and_leave_the_order_out(n, ci, co):
    g = torch.Generator().manual_seed(n)
    flat = torch.randperm(20 ** 3, generator=g)[:n]
    coords = torch.stack([torch.zeros_like(flat), flat // 400, flat // 20 % 20, flat % 20], 1).int().cuda()
    shape = torch.Size([1, ci, 20, 20, 20])
    feats, weight = torch.randn(n, ci, generator=g).half().cuda(), (torch.randn(co, 3, 3, 3, ci, generator=g) / (27 * ci) ** 0.5).half().cuda()
    bias = torch.randn(co, generator=g).half().cuda()
    with torch.no_grad():
        out, cache = sparse_submanifold_conv3d(feats, coords, shape, weight, bias)
        clamped, _ = sparse_submanifold_conv3d_relu(feats, coords, shape, weight, bias, neighbor_cache=cache)
    assert "sorted_idx" not in cache.__dict__ and torch.equal(clamped, torch.relu(out))
    padded = (ci + 7) // 8 * 8
    f, w = torch.zeros(n, padded).half().cuda(), torch.zeros(co, 27, padded).half().cuda()
    f[:, :ci], w[:, :, :ci] = feats, weight.view(co, 27, ci)
    assert torch.equal(out, few(f, w, bias, cache["neighbor_map"].view(torch.int32), 0))
    trained, _ = sparse_submanifold_conv3d(feats.clone().requires_grad_(), coords, shape, weight.clone().requires_grad_(), bias, neighbor_cache=cache)
    assert float((trained.detach() - out).abs().max()) <= 4e-3 * float(out.abs().max())


def test_where_it_holds():
    pays = nat.lib().fgx_conv_gemm_few_pays
    f16, f32 = nat.DTYPE_CODE[torch.float16], nat.DTYPE_CODE[torch.float32]
    assert pays(f16, nat.sz(864), 32, 32, 27) and pays(f16, nat.sz(20000), 24, 32, 27) and pays(f16, nat.sz(500), 128, 64, 8)
    assert not pays(f32, nat.sz(864), 32, 32, 27) and not pays(f16, nat.sz(0), 32, 32, 27) and not pays(f16, nat.sz(864), 30, 32, 27)
    assert not pays(f16, nat.sz(864), 40, 40, 27) and not pays(f16, nat.sz(40000), 32, 32, 27) and not pays(f16, nat.sz(500), 136, 64, 8)
