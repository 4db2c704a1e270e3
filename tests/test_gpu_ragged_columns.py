"""16-bit layers of ragged channel counts over rows enough for the kernels of whole 16-byte pieces (first layers, resident rows): the general
kernels' sums, cut to the channels that are there."""
import pytest
import torch

from flexgemm_amd.ops import spconv
from flexgemm_amd.ops.spconv import sparse_conv3d_relu, sparse_submanifold_conv3d, sparse_submanifold_conv3d_relu
from flexgemm_amd.workloads import reference_test_shell

pytestmark = pytest.mark.gpu


# below and above the rows from which they are taken (131 072 under more than 32 columns, else 393 216); up to one piece, two, four, beyond
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("res,ci,co", [(64, 5, 41), (190, 5, 41), (190, 19, 27), (320, 11, 11), (320, 19, 27), (320, 30, 19), (320, 24, 20), (320, 33, 7)])
def test_against_sums_in_64_bits(dtype, res, ci, co):
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    n, shape = len(coords), torch.Size([1, ci, res, res, res])
    print(f"[case] {n} rows {ci}->{co} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(ci)
    feats = torch.randn(n, ci, generator=g, device="cuda").to(dtype).requires_grad_(True)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5).to(dtype).requires_grad_(True)
    bias = torch.randn(co, generator=g, device="cuda").to(dtype).requires_grad_(True)
    up = torch.randn(n, co, generator=g, device="cuda").to(dtype)
    out, cache = sparse_submanifold_conv3d_relu(feats, coords, shape, weight, bias)
    grads = torch.autograd.grad(out, [feats, weight, bias], up)
    with torch.no_grad():       # the pass that records nothing adds in the same order
        again, _ = sparse_submanifold_conv3d_relu(feats, coords, shape, weight, bias, cache)
    assert out.shape == (n, co) and out.is_contiguous() and torch.equal(out, again)
    m = cache.neighbor_map.view(torch.int32)
    x, w, u = feats.detach().double(), weight.detach().double().reshape(co, 27, ci), up.double() * (out.detach() > 0)
    want, gx, gw = bias.detach().double().repeat(n, 1), torch.zeros(n, ci, dtype=torch.double, device="cuda"), torch.zeros(co, 27, ci, dtype=torch.double, device="cuda")
    for v in range(27):
        r = (m[:, v] >= 0).nonzero()[:, 0]
        s = m[r, v].long()
        want[r] += x[s] @ w[:, v].t().contiguous()
        gx.index_add_(0, s, u[r] @ w[:, v])
        gw[:, v] = u[r].t().contiguous() @ x[s]
    # one rounding to the type
    for got, exact in ((out, want.relu()), (grads[0], gx), (grads[1].reshape(co, 27, ci), gw), (grads[2], u.sum(0))):
        assert got.shape == exact.shape
        assert float((got.detach().double() - exact).norm() / exact.norm()) <= torch.finfo(dtype).eps / 2


def _sums(m, src, weight, rows):
    """64-bit sums of src's rows through a map [rows, V] and the weight [V, K, columns]."""
    out = torch.zeros(rows, weight.shape[2], dtype=torch.double, device="cuda")
    for v in range(m.shape[1]):
        r = (m[:, v] >= 0).nonzero()[:, 0]
        out[r] += src[m[r, v].long()] @ weight[v].contiguous()
    return out


# A generic convolution, whose input gradient goes through a map of its own (offsets as they are): outputs of ragged first layers (5 -> 41), input gradients of
# ragged columns (13 -> 11 and 41 -> 11), both; more and fewer rows than either limit, more outputs than inputs and fewer
@pytest.mark.parametrize("res,ci,co,stride", [(190, 5, 41, 1), (320, 5, 41, 2), (190, 41, 11, 1), (320, 41, 11, 2), (320, 13, 11, 2), (64, 13, 11, 1)])
def test_generic_convolution(res, ci, co, stride):
    dtype = torch.bfloat16
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    n, shape = len(coords), torch.Size([1, ci, res, res, res])
    print(f"[case] {n} rows {ci}->{co} stride {stride}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(ci)
    feats = torch.randn(n, ci, generator=g, device="cuda").to(dtype).requires_grad_(True)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5).to(dtype).requires_grad_(True)
    bias = torch.randn(co, generator=g, device="cuda").to(dtype).requires_grad_(True)
    geometry = dict(stride=(stride,) * 3, padding=(1, 1, 1))
    out, out_coords, cache = sparse_conv3d_relu(feats, coords, shape, weight, bias, **geometry)
    up = torch.randn(len(out_coords), co, generator=g, device="cuda").to(dtype)
    grads = torch.autograd.grad(out, [feats, weight, bias], up)
    m, back = cache.neighbor_map.view(torch.int32), cache.neighbor_map_bwd.view(torch.int32)
    x, w, u = feats.detach().double(), weight.detach().double().reshape(co, 27, ci), up.double() * (out.detach() > 0)
    want = _sums(m, x, w.permute(1, 2, 0), len(m)) + bias.detach().double()
    gx = _sums(back, u, w.permute(1, 0, 2), n)
    gw = torch.zeros(co, 27, ci, dtype=torch.double, device="cuda")
    for v in range(27):
        r = (m[:, v] >= 0).nonzero()[:, 0]
        gw[:, v] = u[r].t().contiguous() @ x[m[r, v].long()]
    for got, exact in ((out, want.relu()), (grads[0], gx), (grads[1].reshape(co, 27, ci), gw), (grads[2], u.sum(0))):
        assert got.shape == exact.shape and got.is_contiguous()
        assert float((got.detach().double() - exact).norm() / exact.norm()) <= torch.finfo(dtype).eps / 2       # one rounding to the type


# Inference on a kept cache, with the packed weight kept too: passes after the one that earned a plan or filled the panel give its bits, and a changed
# weight gives the new one's
@pytest.mark.parametrize("panels", [False, True])
@pytest.mark.parametrize("res,ci,co", [(190, 5, 41), (320, 11, 11), (320, 24, 20), (320, 40, 20)])
def test_kept_cache_in_inference(res, ci, co, panels):
    dtype = torch.float16
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    n, shape = len(coords), torch.Size([1, ci, res, res, res])
    print(f"[case] {n} rows {ci}->{co} panels {panels}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(co)
    feats = torch.randn(n, ci, generator=g, device="cuda").to(dtype)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5).to(dtype)
    bias = torch.randn(co, generator=g, device="cuda").to(dtype)
    spconv.set_weight_panel_cache(panels)
    try:
        with torch.no_grad():
            first, cache = sparse_submanifold_conv3d(feats, coords, shape, weight, bias)
            m = cache.neighbor_map.view(torch.int32)
            for scale in (1.0, -2.0):
                weight *= scale
                want = _sums(m, feats.double(), weight.double().reshape(co, 27, ci).permute(1, 2, 0), n) + bias.double()
                outs = [sparse_submanifold_conv3d(feats, coords, shape, weight, bias, cache)[0] for _ in range(6)]
                for out in outs:
                    assert out.shape == (n, co) and out.is_contiguous()
                    assert float((out.double() - want).norm() / want.norm()) <= torch.finfo(dtype).eps / 2
                assert all(torch.equal(out, outs[-1]) for out in outs[-3:])
    finally:
        spconv.set_weight_panel_cache(False)
