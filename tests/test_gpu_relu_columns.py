"""The gradient of a ReLU from its output, rows filled up; layers of ragged channel counts with and without the filled rows kept."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import sparse_submanifold_conv3d, sparse_submanifold_conv3d_relu
from flexgemm_amd.workloads import reference_test_shell

pytestmark = pytest.mark.gpu


# whole and ragged 16-byte pieces, odd and even element counts, one row and many, rows that start on no word
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols,out_cols,skip", [(1, 1, 8, 0), (300, 82, 88, 0), (301, 7, 7, 0), (77, 130, 136, 1), (5, 8, 8, 0), (70000, 9, 16, 0), (33, 20, 21, 0)])
def test_relu_columns(dtype, rows, cols, out_cols, skip):
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    grad = torch.randn(rows * cols + skip, generator=g, device="cuda").to(dtype)[skip:].view(rows, cols)
    y = torch.relu(torch.randn(rows * cols + skip, generator=g, device="cuda").to(dtype)[skip:].view(rows, cols))
    flat = y.view(-1)
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), -0.0, 0.0, float(torch.finfo(dtype).tiny) / 4, -1.0], device="cuda").to(dtype)
    flat[:min(7, flat.numel())] = special[:min(7, flat.numel())]
    grad.view(-1)[-1] = float("nan")
    out = torch.full((rows, out_cols), 7.0, device="cuda").to(dtype)
    nat.check(nat.lib().fgx_relu_columns(C.c_int(nat.DTYPE_CODE[dtype]), nat.ptr(grad), nat.ptr(y), nat.sz(rows), C.c_int(cols), nat.ptr(out), C.c_int(out_cols),
                                         nat.stream()))
    want = torch.where(y > 0, grad, torch.zeros((), dtype=dtype, device="cuda"))
    assert torch.equal(out[:, :cols].nan_to_num(nan=3.0), want.nan_to_num(nan=3.0)) and not out[:, cols:].any()


@pytest.mark.parametrize("dtype,ci,co", [(torch.float16, 82, 82), (torch.bfloat16, 6, 41), (torch.float16, 130, 64), (torch.float32, 33, 66)])
@pytest.mark.parametrize("relu", [False, True])
def test_filled_rows_change_nothing(dtype, ci, co, relu):
    coords = torch.from_numpy(reference_test_shell(12)).cuda()
    n, shape = len(coords), torch.Size([1, ci, 12, 12, 12])
    g = torch.Generator(device="cuda").manual_seed(ci)
    feats = torch.randn(n, ci, generator=g, device="cuda").to(dtype).requires_grad_(True)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / 30).to(dtype).requires_grad_(True)
    bias = torch.randn(co, generator=g, device="cuda").to(dtype).requires_grad_(True)
    up = torch.randn(n, co, generator=g, device="cuda").to(dtype)

    def grads(composed=False, twice=False):
        op = sparse_submanifold_conv3d_relu if relu and not composed else sparse_submanifold_conv3d
        out, _ = op(feats, coords, shape, weight, bias)
        out = torch.relu(out) if relu and composed else out
        first = torch.autograd.grad(out, [feats, weight, bias], up, retain_graph=twice)
        return torch.autograd.grad(out, [feats, weight, bias], up) if twice else first

    want = grads()
    with torch.autograd.graph.save_on_cpu():        # (keeps no filled rows)
        other = grads()
    for a, b, c, d in zip(want, other, grads(twice=True), grads(composed=True)):
        assert a.shape == b.shape and torch.equal(a, b) and torch.equal(a, c) and torch.equal(a, d)


# What a layer holds between its passes beside its output: up to 256 MB of filled rows, nothing to speak of where they are more
@pytest.mark.parametrize("res,ci,kept", [(60, 82, True), (500, 130, True), (510, 130, False), (510, 131, False)])
def test_memory_held_between_the_passes(res, ci, kept):
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    n, shape, co = len(coords), torch.Size([1, ci, res, res, res]), 64
    feats = torch.randn(n, ci, device="cuda").half().requires_grad_(True)
    weight = (torch.randn(co, 3, 3, 3, ci, device="cuda") / 30).half().requires_grad_(True)
    filled = n * ((ci + 7) // 8 * 8) * 2
    assert (filled <= 256 << 20) == kept
    out, cache = sparse_submanifold_conv3d(feats, coords, shape, weight)
    torch.autograd.grad(out, [feats, weight], torch.ones_like(out))         # (the cache has all of its tables)
    del out
    before = torch.cuda.memory_allocated()
    out, _ = sparse_submanifold_conv3d(feats, coords, shape, weight, None, cache)
    held = torch.cuda.memory_allocated() - before - out.untyped_storage().nbytes()
    assert held <= (filled if kept else 0) + (1 << 20)
    torch.autograd.grad(out, [feats, weight], torch.ones_like(out))
