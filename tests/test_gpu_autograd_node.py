"""The operators' native autograd node under what autograd offers around a node: hooks of the saved tensors, recomputation,
refusal of what it does not differentiate, graphs thousands of layers deep."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.utils.checkpoint import checkpoint

import flex_gemm
from flexgemm_amd.ops.spconv import submanifold_conv3d as impl
from flexgemm_amd.workloads import reference_test_shell

spconv = flex_gemm.ops.spconv
pytestmark = pytest.mark.gpu


def _layer(device, relu, c=32):
    gen = torch.Generator(device=device).manual_seed(5)
    coords = torch.from_numpy(reference_test_shell(16)).to(device)
    shape = torch.Size([1, c, 16, 16, 16])
    feats = torch.randn(coords.shape[0], c, generator=gen, device=device).half().requires_grad_()
    weight = (torch.randn(c, 3, 3, 3, c, generator=gen, device=device) / 30).half().requires_grad_()
    bias = torch.randn(c, generator=gen, device=device).half().requires_grad_()
    op = spconv.sparse_submanifold_conv3d_relu if relu else spconv.sparse_submanifold_conv3d
    cache = op(feats, coords, shape, weight, bias)[1]
    return lambda f, w, b: op(f, coords, shape, w, b, cache)[0], (feats, weight, bias)


def _same(a, b):
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("relu,saved", [(False, 3), (True, 4)])
def test_saved_tensor_hooks_see_every_saved_tensor(gpu_device, relu, saved):
    layer, leaves = _layer(gpu_device, relu)
    out = layer(*leaves)
    up = torch.ones_like(out)
    plain = torch.autograd.grad(out, leaves, up)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(gpu_device)):
        out = layer(*leaves)
    _same(torch.autograd.grad(out, leaves, up), plain)
    assert len(packed) == saved


@pytest.mark.parametrize("relu", [False, True])
def test_recomputed_in_the_backward_pass(gpu_device, relu):
    layer, leaves = _layer(gpu_device, relu)
    out = layer(*leaves)
    up = torch.ones_like(out)
    plain = torch.autograd.grad(out, leaves, up)
    again = checkpoint(lambda *a: layer(*a), *leaves, use_reentrant=False)
    _same(torch.autograd.grad(again, leaves, up), plain)


def test_what_is_not_differentiated_is_refused(gpu_device):
    layer, (feats, weight, bias) = _layer(gpu_device, False)
    with forward_ad.dual_level(), pytest.raises((NotImplementedError, RuntimeError)):
        layer(forward_ad.make_dual(feats.detach(), torch.ones_like(feats)), weight, bias)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda f: layer(f, weight.detach(), bias.detach()).float().sum())(feats.detach())
    out = layer(feats, weight, bias)
    torch.autograd.grad(out, feats, torch.ones_like(out))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, feats, torch.ones_like(out))
    for changed in (weight, bias):
        out = layer(feats, weight, bias)
        with torch.no_grad():
            changed.add_(1)
        with pytest.raises(RuntimeError, match="inplace"):
            torch.autograd.grad(out, feats, torch.ones_like(out))


def test_a_chain_of_many_layers_is_freed(gpu_device):
    layer, (h, weight, bias) = _layer(gpu_device, False, c=8)
    for _ in range(20000):
        h = layer(h, weight, bias)
    del h


@pytest.mark.parametrize("c", [8, 64])
def test_arguments_that_do_not_fit_the_cache_are_refused(gpu_device, c):
    """On the host, before a kernel runs: the kernels would read past the map or the bias, or another device's memory."""
    coords = torch.from_numpy(reference_test_shell(16)).to(gpu_device)
    shape = torch.Size([1, c, 16, 16, 16])
    feats = torch.zeros(len(coords), c, dtype=torch.half, device=gpu_device)
    weight = torch.zeros(c, 3, 3, 3, c, dtype=torch.half, device=gpu_device)
    cache = spconv.sparse_submanifold_conv3d(feats, coords, shape, weight)[1]

    def call(w, b=None):
        return spconv.sparse_submanifold_conv3d(feats, coords, shape, w, b, cache)

    for other in (torch.zeros(c, 3, 3, 1, c).half().to(gpu_device), weight.cpu()):
        with pytest.raises(ValueError):
            call(other)
    for bias in (torch.zeros(c - 1, dtype=torch.half, device=gpu_device), torch.zeros(c, dtype=torch.half)):
        with pytest.raises(ValueError):
            call(weight, bias)
    with pytest.raises(ValueError):
        impl._wgrad(feats[:-1], feats, cache, 27)
    w = weight.clone().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):          # (kept on the host and left there)
        out = call(w)[0]
    with pytest.raises(ValueError, match="saved tensor"):
        torch.autograd.grad(out, w, torch.ones_like(out))
    torch.autograd.grad(call(w)[0], w, torch.ones_like(out))


def test_errors_of_the_backward_pass_keep_their_type(gpu_device):
    """What a backward pass refuses on the host is refused with the exception that a call outside autograd raises."""
    layer, (feats, weight, bias) = _layer(gpu_device, False)
    coords = torch.from_numpy(reference_test_shell(16)).to(gpu_device)
    full = spconv.SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, 32, 16, 16, 16]), (3, 3, 3), (1, 1, 1), True)
    seg = full.valid_signal_seg.view(torch.int32).clone()
    seg[-1] += 100                                          # names more pairs than the lists hold
    cache = spconv.SubMConv3dNeighborCache(neighbor_map=full.neighbor_map, gray_code=full.gray_code, sorted_idx=full.sorted_idx,
                                           valid_signal_i=full.valid_signal_i, valid_signal_o=full.valid_signal_o,
                                           valid_signal_seg=seg.view(torch.uint32))
    out = spconv.sparse_submanifold_conv3d(feats, coords, torch.Size([1, 32, 16, 16, 16]), weight, bias, cache)[0]
    with pytest.raises(ValueError, match="pair lists"):
        torch.autograd.grad(out, weight, torch.ones_like(out))
