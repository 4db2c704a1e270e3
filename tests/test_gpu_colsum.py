"""Column sums: one thread or many across a row, rows that fill a slice, a thread's unrolled walk, or pass them by one."""
import pytest
import torch

from flexgemm_amd.ops.spconv import submanifold_conv3d as impl


SHAPES = [(1, 1), (7, 300), (8, 300), (17, 257), (129, 255), (16, 1024), (33, 1024), (1024 * 16 + 1, 2048), (1024 * 16 + 9, 301), (257, 8), (1000, 77), (70000, 27)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,cols", SHAPES)
def test_column_sums(gpu_device, dtype, n, cols):
    x = torch.randn(n, cols, generator=torch.Generator().manual_seed(n + cols)).to(dtype)
    got = impl._colsum(x.to(gpu_device)).cpu().double()
    want, size = x.double().sum(0), x.double().abs().sum(0)
    # fp32 sums of n values, rounded once to the type
    bound = min(n, 4096) * 2.0 ** -24 * size + torch.finfo(dtype).eps / 2 * want.abs() + torch.finfo(dtype).tiny
    assert bool(((got - want).abs() <= bound).all())


# Rows that can be counted: whole numbers from -1 to 2 whose column sums stay between 0 and 61, exact in all three types and in any order.  A row left out
# or taken twice shows in two of three columns.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,cols", SHAPES)
def test_every_row_is_added_once(gpu_device, dtype, n, cols):
    gen = torch.Generator().manual_seed(n * cols)
    half = torch.randint(-1, 2, (n // 2, cols), generator=gen)
    x = torch.cat([half, -half[torch.randperm(n // 2, generator=gen)], torch.ones(n % 2, cols, dtype=torch.int64)])
    x[torch.randperm(n, generator=gen)[:60]] += 1
    got = impl._colsum(x.to(dtype).to(gpu_device)).cpu()
    assert torch.equal(got, x.sum(0).to(dtype))
