"""The tiled gather GEMM reading the weight itself against the same kernel on a packed panel: the same products in the same
order, so the same bits; what lies around the weight in memory must not matter."""
import ctypes as C

import pytest
import torch

import flex_gemm
from flexgemm_amd import _native as nat
from flexgemm_amd.workloads import reference_test_shell

spconv = flex_gemm.ops.spconv
pytestmark = pytest.mark.gpu

TILES = [(256, 128, 64), (256, 128, 128), (128, 128, 64), (128, 64, 64), (128, 32, 64), (64, 64, 64), (64, 32, 64), (32, 32, 64)]


def _panel(weight, mode, sched):
    co, v, ci = weight.shape
    code = nat.DTYPE_CODE[weight.dtype]
    L = nat.lib()
    args = [C.c_int(code), C.c_int(mode)]
    nbytes = L.fgx_weight_panel_bytes(*args, C.c_int(ci), C.c_int(co), C.c_int(v), C.c_int(sched.slab_bytes), C.c_int(sched.tile_cols))
    panel = torch.empty(nbytes, dtype=torch.uint8, device=weight.device)
    nat.check(L.fgx_pack_weight(*args, nat.ptr(weight), C.c_int(ci), C.c_int(co), C.c_int(v), C.c_int(sched.slab_bytes),
                                C.c_int(sched.tile_cols), nat.ptr(panel), nat.stream()))
    return panel


# channels that end inside a slab, inside a tile and on their edges; one piece; more columns than rows and the reverse
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ci,co", [(8, 8), (64, 64), (72, 136), (264, 40), (128, 320), (72, 15), (296, 295)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_weight_read_in_place_gives_the_panel_products(gpu_device, monkeypatch, tile, ci, co, dtype):
    print(f"[case] tile={tile} ci={ci} co={co} {dtype}", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    coords = torch.from_numpy(reference_test_shell(12)).to(gpu_device)
    n = coords.shape[0]
    cache = spconv.SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 12, 12, 12]), (3, 3, 3), (1, 1, 1), True)
    room = torch.full((co * 27 * ci + 4096,), float("nan"), dtype=dtype, device=gpu_device)
    weight = room[2048:2048 + co * 27 * ci].view(co, 27, ci)
    weight.copy_(torch.randn(co, 27, ci, generator=gen, device=gpu_device) / 30)
    real = nat.table_lookup
    for mode in (0, 1, 2) if dtype != torch.float32 and co % 8 == 0 else (0,):
        sched = real(0, dtype, n, ci, co, 27)
        sched.tile_rows, sched.tile_cols, sched.slab_bytes, sched.stream = *tile, 0
        assert nat.lib().fgx_conv_gather_gemm_weight_pays(C.c_int(nat.DTYPE_CODE[dtype]), C.c_int(mode), C.c_int(ci), C.c_int(co), C.c_int(27))
        src = torch.randn(n, ci if mode == 0 else co, generator=gen, device=gpu_device).to(dtype)
        bias = torch.randn(co, generator=gen, device=gpu_device).to(dtype) if mode == 0 else None
        panel = _panel(weight, mode, sched)
        for splitk in (1, 3):
            sched.splitk = splitk
            monkeypatch.setattr(nat, "table_lookup", lambda *a, **k: sched)
            for masked in (True, False):
                want = nat.host().gather_gemm(src, weight, bias, cache, mode, True, masked, 0, False, panel)[0]
                got = nat.host().gather_gemm(src, weight, bias, cache, mode, True, masked, 0, False, None)[0]
                assert torch.isfinite(want).all() and torch.equal(got, want), (mode, splitk, masked)


def test_shapes_that_need_a_panel(gpu_device):
    def pays(*a):
        return bool(nat.lib().fgx_conv_gather_gemm_weight_pays(*[C.c_int(x) for x in a]))

    f16, f32 = nat.DTYPE_CODE[torch.float16], nat.DTYPE_CODE[torch.float32]
    assert pays(f16, 1, 8, 16, 27) and pays(f32, 0, 4, 4, 27)
    assert not pays(f16, 0, 12, 16, 27) and not pays(f16, 1, 16, 12, 27) and pays(f16, 0, 16, 12, 27)      # no whole 16-byte pieces
    assert not pays(f32, 1, 64, 64, 27)                                        # transposing reads are 16 bits wide
    assert not pays(f16, 0, 8192, 8192, 27)                                    # past 32-bit offsets
