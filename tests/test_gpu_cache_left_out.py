"""A cache that a layer builds for itself without the tables its kernels do not read: the same tables once somebody asks, the same
results of other layers on it."""
import pytest
import torch

import flex_gemm
from flexgemm_amd.ops.spconv.submanifold_conv3d import SubMConv3dFunction
from flexgemm_amd.workloads import reference_test_shell

spconv = flex_gemm.ops.spconv
pytestmark = pytest.mark.gpu


def _layer(c_in, c_out, n, dtype, device, gen):
    w = (torch.randn(c_out, 3, 3, 3, c_in, generator=gen, device=device) / 30).to(dtype).requires_grad_(True)
    f = torch.randn(n, c_in, generator=gen, device=device).to(dtype).requires_grad_(True)
    return f, w


def _bits(t):
    return t.view(torch.int32) if t.dtype == torch.uint32 else t


# a first layer, the resident-row kernels (from 32 768 rows on a grid that walks), the products over pairs -- whose weight gradient reads the lists
@pytest.mark.parametrize("res,ci,co,dtype,lists", [(40, 8, 48, torch.bfloat16, False), (224, 32, 16, torch.float16, False),
                                                   (16, 256, 256, torch.bfloat16, True), (24, 64, 64, torch.float32, True)])
def test_tables_that_a_layer_does_not_read(gpu_device, res, ci, co, dtype, lists):
    gen = torch.Generator(device=gpu_device).manual_seed(res)
    coords = torch.from_numpy(reference_test_shell(res)).to(gpu_device)
    n, shape = coords.shape[0], torch.Size([1, ci, res, res, res])
    f, w = _layer(ci, co, n, dtype, gpu_device, gen)
    if ci == 8:
        f = f.detach()                                  # (a network's input)
    whole = SubMConv3dFunction._compute_neighbor_cache(coords, shape, (3, 3, 3), (1, 1, 1), True)
    assert "sorted_idx" in whole.__dict__ and "valid_signal_seg" in whole.__dict__

    def step(feats, weight, cache):
        out, cache = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight, None, cache)
        return [out, *torch.autograd.grad(out, [t for t in (feats, weight) if t.requires_grad], torch.ones_like(out))], cache

    got, cache = step(f, w, None)
    assert "sorted_idx" not in cache.__dict__ and ("valid_signal_seg" in cache.__dict__) == lists
    want, _ = step(f, w, whole)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    # another kind of layer on the same cache: whatever it reads is made on the way
    f2, w2 = _layer(128, 128, n, torch.float16, gpu_device, gen)
    for a, b in zip(step(f2, w2, cache)[0], step(f2, w2, whole)[0]):
        assert torch.equal(a, b)
    assert "sorted_idx" in cache.__dict__ and "valid_signal_seg" in cache.__dict__
    for name in ("neighbor_map", "gray_code", "sorted_idx", "valid_signal_seg", "valid_signal_i", "valid_signal_o"):
        assert torch.equal(_bits(cache[name]), _bits(whole[name])), name
    # ... and a reader of the fields
    _, fresh = step(f, w, None)
    assert torch.equal(fresh.sorted_idx, whole.sorted_idx) and torch.equal(_bits(fresh["valid_signal_i"]), _bits(whole.valid_signal_i))
    with torch.no_grad():
        _, inference = spconv.sparse_submanifold_conv3d(f, coords, shape, w, None, None)
    assert not hasattr(inference, "valid_signal_i") and torch.equal(inference.sorted_idx, whole.sorted_idx)
