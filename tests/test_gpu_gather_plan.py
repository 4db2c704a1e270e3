"""The gather plan of a row order with its tables and item order, made at once (few tiles) and in separate launches (many)."""
import ctypes as C

import numpy as np
import pytest
import torch

from flexgemm_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tile_rows", [(1, 128), (63, 64), (129, 128), (5000, 256), (5000, 100), (3000, 512), (700, 1024), (4096 * 64, 64), (4096 * 64 + 1, 64)])
@pytest.mark.parametrize("v", [8, 27, 32])
@pytest.mark.parametrize("col_tiles", [0, 1, 3])
def test_plan_against_numpy(n, tile_rows, v, col_tiles):
    rng = np.random.default_rng(n + v)
    nmap = rng.integers(0, n, (n, v)).astype(np.uint32)
    nmap[rng.random((n, v)) < 0.6] = 0xFFFFFFFF
    nmap[rng.random(n) < 0.2] = 0xFFFFFFFF
    nmap[:tile_rows] = 0xFFFFFFFF if n > 2000 else nmap[:tile_rows]             # a tile without any offset
    order = rng.permutation(n).astype(np.int64)
    if n > 2000:
        order = np.arange(n, dtype=np.int64)
    gray = ((nmap != 0xFFFFFFFF) << np.arange(v, dtype=np.int64)).sum(1).astype(np.uint32)
    nt = -(-n // tile_rows)
    padded = np.concatenate([order, np.full(nt * tile_rows - n, -1)]).reshape(nt, tile_rows)
    code = np.bitwise_or.reduce(np.where(padded >= 0, gray[padded], np.uint32(0)), axis=1).astype(np.uint32)
    present = ((code[:, None] >> np.arange(v, dtype=np.uint32)) & 1).astype(np.int64)
    seg = np.concatenate([[0], np.cumsum(present.sum(1))])
    plan_seg = np.concatenate([[0], np.cumsum(np.maximum(present.sum(1), 1))])
    cuda = lambda a: torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda()
    d_map, d_order, d_gray = cuda(nmap), cuda(order), cuda(gray)
    d_code = torch.empty(nt, dtype=torch.int32, device="cuda")
    d_seg, d_plan = (torch.full((nt + 2,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
    d_idx = torch.full((int(plan_seg[-1]) + 1, tile_rows), -7, dtype=torch.int32, device="cuda")
    d_band = torch.full((int(plan_seg[-1]) + 1,), -7, dtype=torch.int32, device="cuda")
    groups, slabs = 256, 2
    L = nat.lib()
    items, ws = None, None
    if col_tiles:
        items = torch.full((nt * col_tiles + 1,), -7, dtype=torch.int32, device="cuda")
        ws = nat.workspace(L.fgx_gather_item_order_workspace_bytes(nat.sz(nt), C.c_int(col_tiles)), torch.device("cuda"))
    nat.check(L.fgx_tile_plan(nat.ptr(d_gray), nat.ptr(d_order), nat.ptr(d_map), nat.sz(n), C.c_int(v), C.c_int(tile_rows), C.c_int(0), nat.ptr(d_code),
                              nat.ptr(d_seg), nat.ptr(d_plan), nat.ptr(d_idx), nat.ptr(d_band), C.c_int(max(col_tiles, 1)), C.c_int(slabs),
                              C.c_int(groups), nat.ptr(ws), nat.ptr(items), nat.stream()))
    assert np.array_equal(d_code.cpu().numpy().view(np.uint32), code)
    assert np.array_equal(d_seg.cpu().numpy(), np.append(seg, -7)) and np.array_equal(d_plan.cpu().numpy(), np.append(plan_seg, -7))
    got_idx, got_band = d_idx.cpu().numpy().view(np.uint32), d_band.cpu().numpy().view(np.uint32)
    safe = np.where(padded >= 0, padded, 0)
    for t in ([0, nt // 2, nt - 1] if nt > 200 else range(nt)):
        rows = np.where((padded[t] >= 0)[:, None], nmap[safe[t]], np.uint32(0xFFFFFFFF))
        offs = np.flatnonzero(present[t])
        if len(offs) == 0:
            assert (got_idx[plan_seg[t]] == 0xFFFFFFFF).all() and got_band[plan_seg[t]] == 0
        for k, o in enumerate(offs):
            assert np.array_equal(got_idx[plan_seg[t] + k], rows[:, o])
            bands = [(rows[b:b + 32, o] != 0xFFFFFFFF).any() for b in range(0, tile_rows, 32)]
            assert got_band[plan_seg[t] + k] == sum(int(x) << b for b, x in enumerate(bands))
    assert (got_idx[-1] == 0xFFFFFFF9).all() and got_band[-1] == 0xFFFFFFF9
    again = torch.full_like(d_idx, -7)
    band2 = torch.full_like(d_band, -7)
    nat.check(L.fgx_gather_plan_fill(nat.ptr(d_map), nat.ptr(d_order), nat.ptr(d_code), nat.ptr(d_plan), nat.sz(n), C.c_int(v), C.c_int(tile_rows),
                                     nat.ptr(again), nat.ptr(band2), nat.stream()))
    assert torch.equal(again, d_idx) and torch.equal(band2, d_band)
    if col_tiles:
        alone = torch.full_like(items, -7)
        nat.check(L.fgx_gather_item_order(nat.ptr(d_code), nat.sz(nt), C.c_int(col_tiles), C.c_int(slabs), C.c_int(groups), nat.ptr(ws), nat.sz(ws.numel()),
                                          nat.ptr(alone), nat.stream()))
        assert torch.equal(items, alone) and np.array_equal(np.sort(items.cpu().numpy()[:-1]), np.arange(nt * col_tiles))
