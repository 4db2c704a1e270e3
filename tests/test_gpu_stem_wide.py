"""First layers into many columns: the product's 256 columns a workgroup and the weight gradient's 128, at the edges of their tiles and steps."""
import pytest
import torch

import test_gpu_stem as narrow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 33, 64, 65, 16411])
@pytest.mark.parametrize("cols,v", [(128, 27), (136, 17), (256, 27), (264, 25), (560, 27)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_products(gpu_device, n, cols, v, dtype):
    for mode in (0, 1, 2):
        narrow.test_products_against_the_sum_over_neighbors(gpu_device, n, 8, cols, v, mode, dtype)


@pytest.mark.parametrize("n", [1, 31, 64, 65, 16411])
@pytest.mark.parametrize("co,v", [(64, 27), (72, 17), (128, 27), (136, 25), (264, 27)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_weight_gradient(gpu_device, n, co, v, dtype):
    narrow.test_against_the_sum_over_pairs(gpu_device, n, 8, co, v, dtype)


# an infinity and a NaN in either of a wavefront's two tiles, and in a column tile of their own
def test_infinities_stay_with_their_pairs(gpu_device):
    nmap, feats, grad = narrow._case(gpu_device, 3000, 8, 200, 27, torch.float16)
    grad[7, 3], grad[2999, 40], grad[100, 130] = float("inf"), float("nan"), -float("inf")
    feats.abs_().add_(0.1)
    want, _ = narrow._pairs(nmap, feats, grad)
    got = narrow._run(nmap, feats, grad)[0].cpu().double()
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got.isnan(), want.isnan()) and not want.isfinite().all()
    ok = want.isfinite()
    # one rounding to the type; 3 000 terms of about one in 32 bits
    assert (got - want)[ok].abs().max() <= 2.0 ** -11 * want[ok].abs().max() + 2.0 ** -14


# Workgroups of four and five steps, whose loaders spend most of their time in the prologue: 128 columns leave LDS for three slots of map words, and the
# last words that the prologue asks for go where the first step's were.  The same bits every time, against the sums over pairs.
@pytest.mark.parametrize("n,co", [(2055, 72), (2055, 264), (66000, 128)])
def test_map_words_of_the_first_steps(gpu_device, n, co):
    nmap, feats, grad = narrow._case(gpu_device, n, 8, co, 27, torch.float16)
    want, _ = narrow._pairs(nmap, feats, grad)
    got = [narrow._run(nmap, feats, grad)[0] for _ in range(20)]
    assert all(torch.equal(g, got[0]) for g in got[1:])
    assert (got[0].cpu().double() - want).abs().max() <= 2.0 ** -11 * want.abs().max() + n ** 0.5 * 2.0 ** -21
