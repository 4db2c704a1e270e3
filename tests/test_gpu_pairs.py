"""The gather GEMM over pairs (conv_gemm_pairs.hip): its plan against the map, its products against the definition in 64 bits, at
the edges of its tiles and of what takes it."""
import ctypes as C

import numpy as np
import pytest
import torch

import flex_gemm
from flexgemm_amd import _native as nat
from flexgemm_amd.workloads import reference_test_shell

spconv = flex_gemm.ops.spconv
EMPTY = 0xFFFFFFFF


def _plan(nmap):
    n, v = nmap.shape
    plan = torch.full((nat.lib().fgx_pair_plan_words(nat.sz(n), C.c_int(v)),), 0x55555555, dtype=torch.int32, device=nmap.device)
    nat.check(nat.lib().fgx_pair_plan(nat.ptr(nmap), nat.sz(n), C.c_int(v), nat.ptr(plan), nat.stream()))
    return plan


def _map(n, n_src, v, density, seed):
    """A random map; offset 0 holds every row, the last offset (of several) none."""
    rng = np.random.default_rng(seed)
    m = rng.integers(0, n_src, size=(n, v), dtype=np.uint32)
    m[rng.random((n, v)) >= density] = EMPTY
    m[:, 0] = rng.integers(0, n_src, size=n)
    if v > 1:
        m[:, -1] = EMPTY
    return m


@pytest.mark.gpu
@pytest.mark.parametrize("n,v", [(1, 1), (1, 27), (63, 8), (1024, 27), (1025, 32), (4096, 27), (4097, 27), (66000, 27), (300000, 2), (5000, 8), (5000, 32)])
def test_plan_lists_the_pairs_in_row_order(gpu_device, n, v):
    m = _map(n, n, v, 0.4, n + v)
    plan = _plan(torch.from_numpy(m.view(np.int32)).view(torch.uint32).to(gpu_device)).cpu().numpy().view(np.uint32)
    counts, place, rows = plan[:32], plan[32:32 + n * v].reshape(n, v), plan[32 + n * v:32 + 2 * n * v].reshape(v, n)
    for o in range(v):
        have = np.flatnonzero(m[:, o] != EMPTY)
        assert counts[o] == len(have)
        assert np.array_equal(rows[o, :len(have)], m[have, o]) and np.array_equal(place[have, o], np.arange(len(have)))
        assert (place[m[:, o] == EMPTY, o] == EMPTY).all()


# 1 ... 129 pairs: one tile and a tile of one pair more; channels of one 16-byte piece, ending inside a slab, a tile, a 32-column block and
# on their edges; one offset, 27, the most
@pytest.mark.gpu
@pytest.mark.parametrize("n,n_src,v", [(1, 3, 1), (127, 50, 27), (128, 200, 8), (129, 129, 27), (700, 300, 32), (2600, 2600, 27)])
@pytest.mark.parametrize("ci,co", [(8, 8), (64, 64), (72, 136), (264, 96), (128, 200), (40, 296)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_products_match_the_definition(gpu_device, n, n_src, v, ci, co, dtype):
    print(f"[case] n={n} n_src={n_src} v={v} {ci}->{co} {dtype}", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(n + ci)
    m = torch.from_numpy(_map(n, n_src, v, 0.45, n).view(np.int32)).to(gpu_device)
    plan = _plan(m.view(torch.uint32))
    L = nat.lib()
    room = torch.full((co * v * ci + 4096,), float("nan"), dtype=dtype, device=gpu_device)      # what lies around the weight must not matter
    weight = room[2048:2048 + co * v * ci].view(co, v, ci)
    weight.copy_(torch.randn(co, v, ci, generator=gen, device=gpu_device) / 8)
    for mode in (0, 1, 2):
        k, cols = (ci, co) if mode == 0 else (co, ci)
        src = torch.randn(n_src, k, generator=gen, device=gpu_device).to(dtype)
        bias = torch.randn(cols, generator=gen, device=gpu_device).to(dtype) if mode == 0 else None
        relu = mode == 0 and dtype != torch.float32
        out = torch.full((n, cols), float("nan"), dtype=dtype, device=gpu_device)
        mask = torch.zeros((n * cols // 8,), dtype=torch.uint8, device=gpu_device) if relu else None
        scratch = torch.full((L.fgx_conv_gemm_pairs_scratch_bytes(nat.sz(n), C.c_int(cols), C.c_int(v)) // 4,), float("nan"), device=gpu_device)
        nat.check(L.fgx_conv_gemm_pairs(C.c_int(nat.DTYPE_CODE[dtype]), C.c_int(mode), nat.ptr(src), nat.ptr(weight), nat.ptr(bias), nat.ptr(plan), nat.sz(n),
                                        nat.sz(n_src), C.c_int(ci), C.c_int(co), C.c_int(v), nat.ptr(scratch), C.c_int(1 if relu else 0), nat.ptr(out),
                                        nat.ptr(mask), nat.stream()))
        want = torch.zeros(n, cols, dtype=torch.float64, device=gpu_device)
        size = torch.zeros_like(want)           # sum of the magnitudes that are added
        for o in range(v):
            have = (m[:, o] != -1).nonzero()[:, 0]
            if not len(have):
                continue
            w = (weight[:, o] if mode == 0 else weight[:, v - 1 - o if mode == 1 else o].T).double().T.contiguous()
            rows = src[m[have, o].long()].double()
            want[have] += rows @ w
            size[have] += rows.abs() @ w.abs()
        if bias is not None:
            want += bias.double()
            size += bias.double().abs()
        if relu:
            want = want.clamp(min=0)
        # one rounding to the result's type, and at most (K + V) roundings of the running sums to 24 bits
        unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
        bound = unit * want.abs() + (k + v) * 2.0 ** -24 * size + 1e-7
        assert ((out.double() - want).abs() <= bound).all(), mode
        if relu:
            bits = (out > 0).view(-1, 8).to(torch.int32)
            assert torch.equal(mask.to(torch.int32), (bits << torch.arange(8, device=gpu_device, dtype=torch.int32)).sum(1).to(torch.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,c", [(torch.float16, 256), (torch.float32, 64)])
def test_operator_takes_it_and_agrees_with_the_masked_kernels(gpu_device, monkeypatch, dtype, c):
    """One plan per map, shared by all layers and both directions."""
    gen = torch.Generator(device=gpu_device).manual_seed(5)
    coords = torch.from_numpy(reference_test_shell(16)).to(gpu_device)
    n = coords.shape[0]
    assert nat.lib().fgx_conv_gemm_pairs_pays(C.c_int(nat.DTYPE_CODE[dtype]), C.c_int(0), nat.sz(n), C.c_int(c), C.c_int(c), C.c_int(27))
    shape = torch.Size([1, c, 16, 16, 16])
    weight = (torch.randn(c, 3, 3, 3, c, generator=gen, device=gpu_device) / 50).to(dtype).requires_grad_(True)
    feats = torch.randn(n, c, generator=gen, device=gpu_device).to(dtype).requires_grad_(True)

    def step():
        out, cache = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight, None, None)
        return out, torch.autograd.grad(out, feats, torch.ones_like(out))[0], cache

    out, grad, cache = step()
    plan = cache.__dict__["_pair_plan"]
    again, _ = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight, None, cache)
    assert cache.__dict__["_pair_plan"] is plan and torch.equal(out, again)
    real = nat.table_lookup
    monkeypatch.setattr(nat, "table_lookup", lambda *a, **k: real(*a, **k))         # (a table of the caller's keeps every shape on it)
    want, want_grad, masked_cache = step()
    assert "_pair_plan" not in masked_cache.__dict__
    unit = {torch.float16: 2.0 ** -10, torch.float32: 1e-5}[dtype]
    for a, b in ((out, want), (grad, want_grad)):
        assert (a - b).abs().max() <= unit * b.abs().max()


@pytest.mark.parametrize("dtype,k,cols,rows", [(torch.float16, 256, 256, 6000), (torch.bfloat16, 512, 512, 6000), (torch.float16, 1024, 64, 6000), (torch.float16, 256, 512, 5000),
                                               (torch.float16, 248, 256, 0), (torch.float16, 256, 56, 0), (torch.float16, 256, 520, 0), (torch.float32, 64, 64, 57600),
                                               (torch.float32, 64, 256, 25720), (torch.float32, 60, 64, 0), (torch.float32, 512, 512, 19418)])
def test_rows_up_to_which_it_is_taken(dtype, k, cols, rows):
    for mode in (0, 1, 2):
        ci, co = (k, cols) if mode == 0 else (cols, k)
        takes = [bool(nat.lib().fgx_conv_gemm_pairs_pays(C.c_int(nat.DTYPE_CODE[dtype]), C.c_int(mode), nat.sz(n), C.c_int(ci), C.c_int(co), C.c_int(27)))
                 for n in (1, rows, rows + 1)]
        assert takes == [rows > 0, rows > 0, False]


# fp32: up to 65 536 rows, 98 304 under at most half as many columns, fewer where the masked kernels pad no slab (64 channels) or hardly a mask (up to
# 8 offsets); the sums' bounds
@pytest.mark.parametrize("k,cols,v,rows", [(64, 64, 27, 57600), (64, 36, 27, 57600), (64, 32, 27, 65536), (64, 8, 27, 65536), (68, 68, 27, 65536), (96, 96, 27, 65536),
                                           (68, 32, 27, 98304), (128, 64, 27, 98304), (128, 68, 27, 65536), (256, 128, 27, 77672), (96, 192, 27, 51440), (96, 96, 9, 65536),
                                           (64, 64, 8, 45000), (64, 32, 8, 45000), (96, 96, 8, 45000), (128, 192, 8, 45000), (96, 48, 8, 65536), (256, 128, 8, 65536)])
def test_rows_up_to_which_fp32_takes_it(k, cols, v, rows):
    for mode in (0, 1, 2):
        ci, co = (k, cols) if mode == 0 else (cols, k)
        takes = [bool(nat.lib().fgx_conv_gemm_pairs_pays(C.c_int(nat.DTYPE_CODE[torch.float32]), C.c_int(mode), nat.sz(n), C.c_int(ci), C.c_int(co), C.c_int(v)))
                 for n in (1, 45000, rows, rows + 1, 98305)]
        assert takes == [True, True, True, False, False]


@pytest.mark.gpu
@pytest.mark.parametrize("ci,co,res", [(72, 72, 110), (128, 64, 156), (64, 64, 118)])
def test_fp32_agrees_with_the_masked_kernels_at_many_rows(gpu_device, monkeypatch, ci, co, res):
    gen = torch.Generator(device=gpu_device).manual_seed(res)
    coords = torch.from_numpy(reference_test_shell(res)).to(gpu_device)
    n = coords.shape[0]
    print(f"[case] {n} rows {ci}->{co}", flush=True)
    shape = torch.Size([1, ci, res, res, res])
    weight = torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device) / (27 * ci) ** 0.5
    feats = torch.randn(n, ci, generator=gen, device=gpu_device).requires_grad_(True)
    up = torch.randn(n, co, generator=gen, device=gpu_device)

    def step():
        out, cache = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight, None, None)
        return out.detach(), torch.autograd.grad(out, feats, up)[0], cache

    out, grad, cache = step()
    assert n > 45000 and "_pair_plan" in cache.__dict__
    real = nat.table_lookup
    monkeypatch.setattr(nat, "table_lookup", lambda *a, **k: real(*a, **k))         # (a table of the caller's keeps every shape on it)
    want, want_grad, other = step()
    assert "_pair_plan" not in other.__dict__
    # 64-bit sums of some rows: 27 ci (27 co) products, each rounded to 2 ** -24 of a sum that stays within the largest output
    some = torch.randperm(n, generator=gen, device=gpu_device)[:2000]
    near = cache.neighbor_map.view(torch.int32)[some].long()
    w64 = weight.detach().reshape(co, 27, ci).double()
    for got, masked, source, panel in ((out, want, feats.detach(), w64.permute(1, 2, 0)), (grad, want_grad, up, w64.flip(1).permute(1, 0, 2))):
        exact = torch.zeros(2000, panel.shape[2], dtype=torch.float64, device=gpu_device)
        for v in range(27):
            exact += (source[near[:, v].clamp(min=0)].double() * (near[:, v:v + 1] >= 0)) @ panel[v].contiguous()
        assert (got[some] - exact).abs().max() <= 1e-5 * exact.abs().max()
        assert (got - masked).abs().max() <= 1e-5 * masked.abs().max()
