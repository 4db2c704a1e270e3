"""The resident-row plan: every table entry names a slot that holds the neighbor's row, or is flagged as not resident."""
import ctypes as C

import numpy as np
import pytest
import torch

from flexgemm_amd import _native as nat

ROWS, SLOTS, STRIDE, HEADER = 128, 448, 32, 256


@pytest.mark.gpu
@pytest.mark.parametrize("v", [1, 9, 27, 31])
@pytest.mark.parametrize("n", [1, 128, 1000])
@pytest.mark.parametrize("spread", [3, 60, 100000])
@pytest.mark.parametrize("own", [0, 1])
def test_plan_names_every_neighbor(v, n, spread, own):
    rng = np.random.default_rng(n * v + spread)
    near = np.arange(n)[:, None] + rng.integers(-spread, spread + 1, (n, v))
    nmap = np.where((near >= 0) & (near < n) & (rng.random((n, v)) < 0.6), near, 0xFFFFFFFF).astype(np.uint32)
    if spread == 100000:
        nmap = rng.integers(0, 4000, (n, v)).astype(np.uint32)              # more distinct sources than slots, or than the hash table
    L = nat.lib()
    size = L.fgx_narrow_plan_bytes(nat.sz(n), C.c_int(v))
    chunks = -(-n // ROWS)
    stride = (size - HEADER) // chunks
    plan = torch.zeros(size, dtype=torch.uint8, device="cuda")
    dev = torch.from_numpy(nmap.view(np.int32)).cuda()
    nat.check(L.fgx_narrow_plan(nat.ptr(dev), None, nat.sz(n), C.c_int(v), C.c_int(own), nat.ptr(plan), nat.stream()))
    raw = plan.cpu().numpy()
    overflowing = 0
    for c in range(chunks):
        one = raw[HEADER + c * stride:HEADER + (c + 1) * stride]
        table = one[:ROWS * STRIDE * 2].view(np.uint16).reshape(ROWS, STRIDE).astype(np.int64)
        sources = one[ROWS * STRIDE * 2:ROWS * STRIDE * 2 + SLOTS * 4].view(np.uint32)
        rows = one[ROWS * STRIDE * 2 + SLOTS * 4:ROWS * STRIDE * 2 + SLOTS * 4 + ROWS * 4].view(np.uint32)
        lo, hi = c * ROWS, min(n, (c + 1) * ROWS)
        assert np.array_equal(rows[:hi - lo], np.arange(lo, hi)) and (rows[hi - lo:] == 0xFFFFFFFF).all()
        want = np.full((ROWS, v), 0xFFFFFFFF, np.uint32)
        want[:hi - lo] = nmap[lo:hi]
        got = table[:, :v]
        lost = got == 0xFFFF
        slot = got >> 6
        assert (slot[(want == 0xFFFFFFFF)] == SLOTS).all()
        held = (want != 0xFFFFFFFF) & ~lost
        assert np.array_equal(sources[slot[held]], want[held]) and ((got[held] >> 4) & 3 == (slot[held] >> 2) & 3).all()
        assert np.array_equal(table[:, STRIDE - 1] != 0, lost.any(1))
        distinct = len(np.unique(np.concatenate([want[want != 0xFFFFFFFF], np.arange(lo, hi, dtype=np.uint32) if own else []])))
        assert lost.any() == (distinct > SLOTS - (ROWS - (hi - lo) if own else 0)) or distinct > SLOTS
        overflowing += bool(lost.any())
    assert raw[:4].view(np.uint32)[0] == overflowing
