"""Up to 32 columns under rows of 256 bytes and more: the streaming kernel from 320 000 voxels, against the tiled kernel on the same map."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import sparse_submanifold_conv3d
from flexgemm_amd.workloads import reference_test_shell


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,cols", [(128, 8), (136, 32), (1024, 16)])
def test_rows_from_which_it_streams(dtype, k, cols):
    for kind, ci, co in ((nat.PASS_FWD, k, cols), (nat.PASS_DGRAD, cols, k)):
        assert [nat.table_lookup(kind, dtype, n, ci, co, 27).stream for n in (319999, 320000, 3000000)] == [0, 1, 1]
        assert nat.table_lookup(kind, dtype, 320000, ci, co, 27).tile_cols == 32
        # few offsets do not pay for its tables
        assert [nat.table_lookup(kind, dtype, 320000, ci, co, v).stream for v in (1, 3, 4, 8, 9)] == ([0, 0, 0, 0, 1] if kind == nat.PASS_DGRAD else [0, 0, 1, 1, 1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ci,co,relu", [(128, 16, False), (168, 24, True), (16, 136, False)])
def test_agrees_with_the_tiled_kernel(gpu_device, monkeypatch, dtype, ci, co, relu):
    res = 288
    coords = torch.from_numpy(reference_test_shell(res)[:320001]).to(gpu_device)
    n = len(coords)
    assert n == 320001
    print(f"[case] {n} rows {ci}->{co} {dtype}", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(ci)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device) / (27 * ci) ** 0.5).to(dtype)
    bias = torch.randn(co, generator=gen, device=gpu_device).to(dtype)
    feats = torch.randn(n, ci, generator=gen, device=gpu_device).to(dtype).requires_grad_(True)
    up = torch.randn(n, co, generator=gen, device=gpu_device).to(dtype)

    def step():
        out, _ = sparse_submanifold_conv3d(feats, coords, torch.Size([1, ci, res, res, res]), weight, bias)
        out = torch.relu(out) if relu else out
        return out.detach(), torch.autograd.grad(out, feats, up)[0]

    got = step()
    real = nat.table_lookup
    monkeypatch.setattr(nat, "table_lookup", lambda kind, dt, rows, *a, **k: real(kind, dt, 300000, *a, **k))
    want = step()
    eps = torch.finfo(dtype).eps
    for a, b, terms in ((got[0], want[0], 27 * ci), (got[1], want[1], 27 * co)):
        # two orders of the same fp32 sums of values below a few, either rounded once to the type
        a, b = a.double(), b.double()
        differ = (a - b).abs() > eps * b.abs() + terms * 2.0 ** -24 * 4
        if relu and terms == 27 * co:        # (a sum that rounds to either side of zero passes its gradient on or not: up to 27 rows see it)
            assert differ.sum() <= 1e-5 * differ.numel()
        else:
            assert not differ.any()
