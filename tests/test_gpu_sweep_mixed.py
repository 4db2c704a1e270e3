"""Weight gradients of 33 ... 64 channels on one side and 65 ... 128 on the other: the sweep's wide tile from 65 536 voxels."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction
from flexgemm_amd.ops.spconv import submanifold_conv3d as impl
from flexgemm_amd.workloads import reference_test_shell


@pytest.mark.parametrize("ci,co", [(33, 65), (64, 128), (128, 40)])
def test_voxels_from_which_it_sweeps(ci, co):
    look = lambda n, v, a=ci, b=co, dt=torch.float16: nat.table_lookup(nat.PASS_WGRAD, dt, n, a, b, v)
    assert [look(n, 27).stream == 2 for n in (8192, 65535, 65536, 1 << 24, (1 << 24) + 1)] == [False, False, True, True, False]
    assert look(65536, 27).tile_rows == look(65536, 27).tile_cols == 128 and look(200000, 8).stream != 2 and look(200000, 9).stream == 2
    assert look(200000, 27, 64, 129).stream != 2 and look(200000, 27, ci, co, torch.float32).stream != 2
    assert look(200000, 27, 64, 64).tile_rows == 64 and look(200000, 27, 65, 128).tile_rows == 128


@pytest.mark.parametrize("ci,co", [(17, 97), (32, 128), (128, 24)])
def test_voxels_from_which_narrow_and_wide_sweep(ci, co):
    look = lambda n, v, a=ci, b=co: nat.table_lookup(nat.PASS_WGRAD, torch.float16, n, a, b, v)
    assert [look(n, 27).stream == 2 for n in (131071, 131072, 1 << 24, (1 << 24) + 1)] == [False, True, True, False] and look(131072, 27).tile_cols == 128
    assert look(200000, 8).stream != 2 and look(200000, 27, 16, 128).stream != 2 and look(200000, 27, 32, 96).stream != 2


@pytest.mark.gpu
@pytest.mark.parametrize("ci,co,dtype,rows", [(40, 128, torch.float16, 65536), (72, 64, torch.bfloat16, 65536), (24, 104, torch.float16, 131072),
                                              (128, 32, torch.bfloat16, 131072)])
def test_agrees_with_the_block_major_kernel(gpu_device, monkeypatch, ci, co, dtype, rows):
    res = 192
    coords = torch.from_numpy(reference_test_shell(res)[:rows + 17]).to(gpu_device)
    n = len(coords)
    assert n == rows + 17
    print(f"[case] {n} rows {ci}->{co} {dtype}", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(ci)
    feats, grad = (torch.randn(n, c, generator=gen, device=gpu_device).to(dtype) for c in (ci, co))
    build = lambda: SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, res, res, res]), (3, 3, 3), (1, 1, 1), True)
    cache = build()
    gw, gb = impl._wgrad(grad, feats, cache, 27, with_bias=True, bias_offset=13)
    assert any(k.startswith("_wgrad_sweep_plan_") for k in vars(cache))
    real, other = nat.table_lookup, build()
    monkeypatch.setattr(nat, "table_lookup", lambda kind, dt, rows, *a, **k: real(kind, dt, 60000, *a, **k))
    want_w, want_b = impl._wgrad(grad, feats, other, 27, with_bias=True, bias_offset=13)
    assert not any(k.startswith("_wgrad_sweep_plan_") for k in vars(other))
    for a, b in ((gw, want_w), (gb, want_b)):
        # two orders of the same fp32 sums of at most n products of random sign, either rounded once to the type
        assert bool(((a.double() - b.double()).abs() <= torch.finfo(dtype).eps * b.double().abs() + 8 * n * 2.0 ** -24).all())
