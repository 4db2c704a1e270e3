"""16-bit layers of ragged channel counts over rows enough for the kernels of whole 16-byte pieces (first layers, resident rows): the general
kernels' sums, cut to the channels that are there."""
import pytest
import torch

from flexgemm_amd.ops.spconv import sparse_submanifold_conv3d_relu
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
