"""The kernels of first layers (8 or 16 channels on the gathered side) against sums over the pairs in 64 bits."""
import pytest
import torch

import flex_gemm
from flexgemm_amd import _native as nat
from flexgemm_amd.workloads import reference_test_shell

spconv = flex_gemm.ops.spconv
pytestmark = pytest.mark.gpu


def _case(device, n, ci, co, v, dtype, seed=1):
    gen = torch.Generator(device=device).manual_seed(seed)
    nmap = torch.randint(0, n, (n, v), generator=gen, device=device)
    nmap[torch.rand(n, v, generator=gen, device=device) < 0.5] = 0xFFFFFFFF
    feats = torch.randn(n, ci, generator=gen, device=device).to(dtype)
    grad = torch.randn(n, co, generator=gen, device=device).to(dtype)
    return nmap.to(torch.uint32), feats, grad


def _run(nmap, feats, grad, with_bias=True):
    import ctypes as C
    n, v, ci, co = *nmap.shape, feats.shape[1], grad.shape[1]
    code, L = nat.DTYPE_CODE[feats.dtype], nat.lib()
    scratch = nat.workspace(L.fgx_wgrad_stem_scratch_bytes(nat.sz(n), C.c_int(ci), C.c_int(co)), feats.device)
    gw = torch.empty(co, v, ci, dtype=feats.dtype, device=feats.device)
    gb = torch.empty(co, dtype=feats.dtype, device=feats.device) if with_bias else None
    nat.check(L.fgx_conv_wgrad_stem(C.c_int(code), nat.ptr(grad), nat.ptr(feats), nat.ptr(nmap), nat.sz(n), C.c_int(ci), C.c_int(co), C.c_int(v),
                                    nat.ptr(scratch), nat.ptr(gw), nat.ptr(gb), nat.stream()))
    return gw, gb


def _pairs(nmap, feats, grad):
    """Per offset, over its pairs alone, in float64 on the CPU."""
    m, f, g = nmap.cpu().to(torch.int64), feats.cpu().double(), grad.cpu().double()
    out = []
    for v in range(m.shape[1]):
        rows = (m[:, v] != 0xFFFFFFFF).nonzero()[:, 0]
        out.append(g[rows].t() @ f[m[rows, v]])
    return torch.stack(out, 1), g.sum(0)


# rows: fewer than a step, one step and one more, a run per workgroup and its remainder; columns: one piece, past one tile
@pytest.mark.parametrize("n", [1, 31, 64, 65, 127, 3716, 16384, 16411, 40003])
@pytest.mark.parametrize("ci,co,v", [(8, 48, 27), (8, 8, 17), (16, 72, 27), (16, 136, 25)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_against_the_sum_over_pairs(gpu_device, n, ci, co, v, dtype):
    print(f"[case] n={n} {ci}->{co} v={v} {dtype}", flush=True)
    nmap, feats, grad = _case(gpu_device, n, ci, co, v, dtype)
    want_w, want_b = _pairs(nmap, feats, grad)
    gw, gb = _run(nmap, feats, grad)
    # one rounding to the type (half an ulp: 2^-11, 2^-8) of sums whose fp32 error is n * 2^-24 of their terms at most
    ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for got, want in ((gw, want_w), (gb, want_b)):
        assert (got.cpu().double() - want).abs().max() <= ulp * want.abs().max() + n ** 0.5 * 2.0 ** -21
    assert torch.equal(_run(nmap, feats, grad, with_bias=False)[0], gw)


def test_infinities_stay_with_their_pairs(gpu_device):
    nmap, feats, grad = _case(gpu_device, 3000, 8, 16, 27, torch.float16)
    grad[7, 3], grad[2999, 5] = float("inf"), float("nan")
    feats.abs_().add_(0.1)
    want, _ = _pairs(nmap, feats, grad)
    got = _run(nmap, feats, grad)[0].cpu().double()
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got.isnan(), want.isnan()) and not want.isfinite().all()
    ok = want.isfinite()
    assert (got - want)[ok].abs().max() <= 2.0 ** -11 * want[ok].abs().max() + 2.0 ** -14


@pytest.mark.parametrize("ci", [3, 8, 16])
def test_operator_takes_it(gpu_device, ci):
    """A first layer through the operator, gradients against torch in float64; the cache is shared with a wider layer."""
    coords = torch.from_numpy(reference_test_shell(20)).to(gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(2)
    n, co = coords.shape[0], 40
    feats = torch.randn(n, ci, generator=gen, device=gpu_device).half()
    weight = (torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device) / 9).half().requires_grad_()
    bias = torch.randn(co, generator=gen, device=gpu_device).half().requires_grad_()
    out, cache = spconv.sparse_submanifold_conv3d(feats, coords, torch.Size([1, ci, 20, 20, 20]), weight, bias)
    up = torch.randn(out.shape, generator=gen, device=gpu_device).half()
    gw, gb = torch.autograd.grad(out, (weight, bias), up)
    want_w, want_b = _pairs(cache.neighbor_map, feats, up)
    assert (gw.cpu().double().view(co, 27, ci) - want_w).abs().max() <= 2.0 ** -11 * want_w.abs().max() + 1e-3
    assert (gb.cpu().double() - want_b).abs().max() <= 2.0 ** -11 * want_b.abs().max() + 1e-3


def _forward(nmap, src, weight, bias, mode, relu, want_mask):
    import ctypes as C
    n, v = nmap.shape
    co, _, ci = weight.shape
    code, L = nat.DTYPE_CODE[src.dtype], nat.lib()
    cols = co if mode == 0 else ci
    out = torch.empty(n, cols, dtype=src.dtype, device=src.device)
    mask = torch.empty(n * cols // 8, dtype=torch.uint8, device=src.device) if want_mask else None
    nat.check(L.fgx_conv_gemm_stem(C.c_int(code), C.c_int(mode), nat.ptr(src), nat.ptr(weight), nat.ptr(bias), nat.ptr(nmap), nat.sz(n), C.c_int(ci),
                                   C.c_int(co), C.c_int(v), C.c_int(1 if relu else 0), nat.ptr(out), nat.ptr(mask), nat.stream()))
    return out, mask


@pytest.mark.parametrize("n", [1, 33, 64, 65, 3716, 16411, 40003])
@pytest.mark.parametrize("k,cols,v", [(8, 48, 27), (8, 8, 17), (8, 136, 27), (16, 72, 27), (16, 200, 25)])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_products_against_the_sum_over_neighbors(gpu_device, n, k, cols, v, mode, dtype):
    print(f"[case] n={n} {k}->{cols} v={v} mode={mode} {dtype}", flush=True)
    ci, co = (k, cols) if mode == 0 else (cols, k)
    nmap, src, _ = _case(gpu_device, n, k, 8, v, dtype)
    gen = torch.Generator(device=gpu_device).manual_seed(9)
    weight = (torch.randn(co, v, ci, generator=gen, device=gpu_device) / 8).to(dtype)
    bias = torch.randn(co, generator=gen, device=gpu_device).to(dtype) if mode == 0 else None
    m = nmap.cpu().to(torch.int64)
    rows = torch.cat([src.cpu().double(), torch.zeros(1, k, dtype=torch.float64)])
    gathered = rows[torch.where(m == 0xFFFFFFFF, n, m)]                       # [n, v, k]
    w = weight.cpu().double()
    w = w if mode == 0 else (w.flip(1) if mode == 1 else w).permute(2, 1, 0)   # [cols, v, k]
    want = gathered.reshape(n, -1) @ w.reshape(cols, -1).t()
    if bias is not None:
        want += bias.cpu().double()
    got, _ = _forward(nmap, src, weight, bias, mode, False, False)
    # one rounding to the type of fp32 sums of at most 432 terms
    ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((got.cpu().double() - want).abs() <= ulp * want.abs() + 1e-4).all()
    relu, bits = _forward(nmap, src, weight, bias, mode, True, True)
    assert torch.equal(relu, got.clamp(min=0))
    on = (bits[:, None] >> torch.arange(8, device=gpu_device)) & 1
    assert torch.equal(on.bool().reshape(n, cols), relu > 0)


def test_a_map_that_starts_between_16_byte_pieces(gpu_device):
    """A hand-made cache whose neighbor map is a row slice of a larger one (rows of 108 bytes): dense, but not on a 16-byte
    boundary, which these kernels' loads need.  The layer runs on the other kernels then."""
    coords = torch.from_numpy(reference_test_shell(20)).to(gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(4)
    n, ci, co = coords.shape[0], 8, 40
    nmap = spconv.SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 20, 20, 20]), (3, 3, 3), (1, 1, 1), False).neighbor_map
    larger = torch.zeros(n + 1, 27, dtype=torch.int32, device=gpu_device)
    larger[1:] = nmap.view(torch.int32)
    cache = spconv.SubMConv3dNeighborCache(neighbor_map=larger[1:].view(torch.uint32))
    assert cache.neighbor_map.is_contiguous() and cache.neighbor_map.data_ptr() % 16
    feats = torch.randn(n, ci, generator=gen, device=gpu_device).half().requires_grad_()
    weight = (torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device) / 9).half().requires_grad_()
    out, _ = spconv.sparse_submanifold_conv3d(feats, coords, torch.Size([1, ci, 20, 20, 20]), weight, None, cache)
    up = torch.randn(out.shape, generator=gen, device=gpu_device).half()
    gf, gw = torch.autograd.grad(out, (feats, weight), up)
    m = nmap.cpu().to(torch.int64)
    w = weight.detach().cpu().double().view(co, 27, ci)

    def through(src, wt):           # [n, v, k] x [cols, v, k]
        rows = torch.cat([src.detach().cpu().double(), torch.zeros(1, src.shape[1], dtype=torch.float64)])
        return rows[torch.where(m == 0xFFFFFFFF, n, m)].reshape(n, -1) @ wt.reshape(wt.shape[0], -1).t()

    want = (through(feats, w), through(up, w.flip(1).permute(2, 1, 0)), _pairs(nmap, feats.detach(), up)[0])
    for got, ref in zip((out.detach(), gf, gw.view(co, 27, ci)), want):
        assert (got.cpu().double() - ref).abs().max() <= 2.0 ** -11 * ref.abs().max() + 1e-3


def _same_classes(got, want):
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got == float("inf"), want == float("inf"))
    assert torch.equal(got == -float("inf"), want == -float("inf"))


# rows with an infinity or NaN among the last of a step, alone in theirs, side by side, over an infinite or zero feature
@pytest.mark.parametrize("ci,co,v,dtype", [(8, 16, 27, torch.float16), (8, 72, 17, torch.bfloat16), (16, 48, 27, torch.bfloat16),
                                           (16, 136, 25, torch.float16)])
def test_infinities_of_many_kinds_stay_with_their_pairs(gpu_device, ci, co, v, dtype):
    print(f"[case] {ci}->{co} v={v} {dtype}", flush=True)
    n = 20011
    nmap, feats, grad = _case(gpu_device, n, ci, co, v, dtype, seed=5)
    inf, nan = float("inf"), float("nan")
    feats[100, 1], feats[101, 2], feats[102, 3] = inf, -inf, 0.0
    m = nmap.view(torch.int32)
    m[64, 3], m[65, 4], m[66, 5], m[70, 3] = 100, 101, 102, 102
    grad[64, 0], grad[65, 1], grad[66, 2], grad[70, 3], grad[n - 1, 4], grad[n - 2, 4], grad[63, 5], grad[5000, 6] = inf, inf, -inf, nan, inf, -inf, -inf, inf
    grad[200:264, 7] = inf
    want_w, want_b = _pairs(nmap, feats, grad)
    gw, gb = _run(nmap, feats, grad)
    for got, want in ((gw.cpu().double(), want_w), (gb.cpu().double(), want_b)):
        _same_classes(got, want)
        ok = want.isfinite()
        # one rounding to the type, sums as in test_against_the_sum_over_pairs
        assert (got - want)[ok].abs().max() <= 2.0 ** (-11 if dtype == torch.float16 else -8) * want[ok].abs().max() + n ** 0.5 * 2.0 ** -21


def test_a_step_that_overflows_everywhere_takes_no_longer(gpu_device):
    """Every element of the gradient infinite, as a step of mixed-precision training with too large a loss scale leaves it."""
    nmap, feats, grad = _case(gpu_device, 200003, 8, 48, 27, torch.bfloat16)

    def fastest(g):
        best = float("inf")
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            _run(nmap, feats, g)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    usual, overflown = fastest(grad), fastest(torch.full_like(grad, float("inf")))
    print(f"[case] {usual:.3f} ms, overflown {overflown:.3f} ms", flush=True)
    assert overflown < 20 * usual


# a first layer with up to 32 columns and more rows than the resident-row kernel asks for: grids that have no cell order, and the
# generic convolution, whose cache has no coordinates, take these kernels at once (nothing of a tile schedule is made)
@pytest.mark.parametrize("generic", [False, True])
@pytest.mark.parametrize("ci,co", [(8, 32), (16, 24)])
def test_narrow_first_layers_without_a_cell_order(gpu_device, generic, ci, co):
    res = 100 if generic else 160
    coords = torch.from_numpy(reference_test_shell(res)).to(gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(6)
    feats = torch.randn(coords.shape[0], ci, generator=gen, device=gpu_device).half()
    weight = (torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device) / 9).half()
    shape = torch.Size([1, ci, res, res, res])
    with torch.no_grad():
        if generic:
            out, _, cache = spconv.sparse_conv3d(feats, coords, shape, weight, None, padding=(1, 1, 1))
        else:
            out, cache = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight)
    assert out.shape[0] >= 32768 and not any(k.startswith(("_plan_", "_mask_code_", "_narrow_plan_buf")) for k in vars(cache))
    m = cache.neighbor_map[::97].cpu().to(torch.int64)
    rows = torch.cat([feats.cpu().double(), torch.zeros(1, ci, dtype=torch.float64)])
    want = rows[torch.where(m == 0xFFFFFFFF, len(feats), m)].reshape(len(m), -1) @ weight.cpu().double().reshape(co, -1).t()
    assert ((out[::97].cpu().double() - want).abs() <= 2.0 ** -11 * want.abs() + 1e-4).all()
