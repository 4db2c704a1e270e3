"""fgx_copy_columns: rows filled up with zeros or cut, every unit and piece width it picks, bit for bit."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("rows,src_cols,dst_cols", [(1, 1, 8), (1000, 6, 8), (777, 5, 8), (3, 7, 16), (1296, 8, 6), (1001, 8, 5), (50, 40, 48), (1, 130003, 130008),
                                                    (300000, 3, 4), (2, 1, 1)])
@pytest.mark.parametrize("offset", [0, 1])
def test_copy_columns(dtype, rows, src_cols, dst_cols, offset):
    bits = torch.int16 if dtype == torch.float16 else torch.int32
    src = torch.randint(-30000, 30000, (offset + rows * src_cols,), device="cuda", dtype=bits)[offset:]
    guarded = torch.full((rows * dst_cols + 16,), 77, device="cuda", dtype=bits)
    nat.check(nat.lib().fgx_copy_columns(C.c_int(src.element_size()), nat.ptr(src), nat.sz(rows), C.c_int(src_cols), nat.ptr(guarded), C.c_int(dst_cols),
                                         nat.stream()))
    want = torch.zeros((rows, dst_cols), device="cuda", dtype=bits)
    both = min(src_cols, dst_cols)
    want[:, :both] = src.view(rows, src_cols)[:, :both]
    assert torch.equal(guarded[:rows * dst_cols].view(rows, dst_cols), want) and bool((guarded[rows * dst_cols:] == 77).all())


def test_refuses_bad_arguments():
    L = nat.lib()
    one = C.c_void_p(4096)
    assert L.fgx_copy_columns(8, one, nat.sz(1), 1, one, 1, None) != 0
    assert L.fgx_copy_columns(4, one, nat.sz(1), 0, one, 1, None) != 0
    assert L.fgx_copy_columns(4, None, nat.sz(1), 1, one, 1, None) != 0
    assert L.fgx_copy_columns(4, C.c_void_p(4098), nat.sz(1), 1, one, 1, None) != 0
    assert L.fgx_copy_columns(4, None, nat.sz(0), 1, None, 1, None) == 0
