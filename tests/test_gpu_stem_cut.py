"""Weight gradient of first layers whose channels were filled up: the true channels' part, and nothing beside it."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat


@pytest.mark.gpu
@pytest.mark.parametrize("ci,out_ci", [(8, 1), (8, 3), (8, 6), (8, 8), (16, 9), (16, 13), (16, 16)])
@pytest.mark.parametrize("n,co,v", [(1, 8, 17), (129, 40, 27), (5000, 136, 25)])
def test_true_channels_of_the_weight_gradient(gpu_device, ci, out_ci, n, co, v):
    gen = torch.Generator(device=gpu_device).manual_seed(n + ci)
    nmap = torch.randint(0, n, (n, v), generator=gen, device=gpu_device)
    nmap[torch.rand(n, v, generator=gen, device=gpu_device) < 0.5] = 0xFFFFFFFF
    nmap = nmap.to(torch.uint32)
    feats, grad = (torch.randn(n, c, generator=gen, device=gpu_device).bfloat16() for c in (ci, co))
    L = nat.lib()
    got = []
    for part in (ci, out_ci):
        scratch = nat.workspace(L.fgx_wgrad_stem_scratch_bytes(nat.sz(n), C.c_int(ci), C.c_int(co)), gpu_device)
        room = torch.full((co * v * part + 2,), 7.0, dtype=torch.bfloat16, device=gpu_device)
        bias = torch.empty(co, dtype=torch.bfloat16, device=gpu_device)
        nat.check(L.fgx_conv_wgrad_stem_cut(C.c_int(nat.DTYPE_CODE[torch.bfloat16]), nat.ptr(grad), nat.ptr(feats), nat.ptr(nmap), nat.sz(n), C.c_int(ci),
                                            C.c_int(part), C.c_int(co), C.c_int(v), nat.ptr(scratch), C.c_void_p(room.data_ptr() + 2), nat.ptr(bias), nat.stream()))
        assert room[0] == 7 and room[-1] == 7
        got.append((room[1:-1].view(co, v, part), bias))
    assert torch.equal(got[1][0], got[0][0][:, :, :out_ci]) and torch.equal(got[1][1], got[0][1])
