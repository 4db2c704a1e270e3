"""Map and plan of the narrow layers from one kernel: the map of the general kernel, and a plan whose every entry names the map's neighbor."""
import ctypes as C

import numpy as np
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.workloads import reference_test_shell

ROWS, SLOTS, STRIDE, HEADER = 128, 448, 32, 256


def _build(coords, dims, dil, walk, plan):
    L, n = nat.lib(), coords.shape[0]
    geom = [C.c_int(int(x)) for x in (*dims, 3, 3, 3, *dil)]
    ws = nat.workspace(L.fgx_subm_cache_grid_workspace_bytes(nat.sz(n), *geom[:4], C.c_int(27), C.c_int(0)), coords.device)
    nmap = torch.full((n, 27), 7, dtype=torch.int32, device=coords.device)
    gray, binary = torch.empty(n, dtype=torch.int32, device=coords.device), torch.empty(n, dtype=torch.int32, device=coords.device)
    none = nat.ptr(None)
    nat.check(L.fgx_subm_cache_build_grid_plan(nat.ptr(coords), nat.sz(n), *geom, C.c_int(0), nat.ptr(ws), nat.sz(ws.numel()), nat.ptr(nmap), nat.ptr(gray),
                                               nat.ptr(binary), none, none, none, none, none, nat.ptr(walk), nat.ptr(plan), nat.stream()))
    return nmap, gray, binary


# rows that fill no chunk, one, one and a row; voxels given twice and outside the grid, which end the walk; a batch; columns that end inside a
# brick; scattered voxels (n = 0).  n < 0: a solid cube of so many cells a side inside the shell, of whose chunks some have more sources than
# slots, and of the last one more than the builder's hash table
@pytest.mark.gpu
@pytest.mark.parametrize("dims,n,extra,dil", [((1, 300, 300, 300), 1, 0, (1, 1, 1)), ((1, 204, 204, 204), 127, 0, (1, 1, 1)), ((1, 204, 204, 204), 128, 0, (2, 1, 16)),
                                              ((3, 205, 210, 131), 129, 0, (1, 1, 1)), ((2, 204, 204, 233), 9000, 700, (1, 1, 1)), ((1, 230, 230, 230), 30000, 0, (1, 2, 3)),
                                              ((1, 230, 230, 230), 0, 0, (1, 1, 1)), ((1, 230, 230, 230), -20, 0, (1, 1, 1)), ((1, 230, 230, 230), -20, 90, (2, 2, 2)),
                                              ((1, 230, 230, 230), -40, 0, (4, 5, 7))])
@pytest.mark.parametrize("order", ["scan", "shuffled"])
def test_plan_beside_the_map(gpu_device, dims, n, extra, dil, order):
    print(f"[case] dims={dims} n={n} extra={extra} dilation={dil} {order}", flush=True)
    rng = np.random.default_rng(abs(n))
    base = reference_test_shell(96) + np.array([0, 50, 3, 30], np.int32)
    base[:, 0] = rng.integers(0, dims[0], len(base))
    solid = n < 0
    if solid:
        side = np.arange(-n, dtype=np.int32) + n // 2
        cube = np.stack(np.meshgrid(0, side + 98, side + 51, side + 78, indexing="ij"), -1).reshape(-1, 4)
        base = np.unique(np.concatenate([base, cube.astype(np.int32)]), axis=0)
    elif n == 0:                                            # no two voxels near each other: every chunk has 128 rows and as many sources
        base = np.unique(rng.integers(0, dims, (4000, 4)).astype(np.int32), axis=0)
    elif n < len(base):
        base = base[:n] if n < 1000 else base[rng.choice(len(base), n, replace=False)]
    base = base[np.lexsort(base.T[::-1])]
    if extra:
        outside = base[:50] + np.array([0, 0, 0, dims[3]], np.int32)
        base = np.concatenate([base, base[rng.integers(0, len(base), extra)], outside])
    if order == "shuffled":
        base = base[rng.permutation(len(base))]
    coords = torch.from_numpy(np.ascontiguousarray(base.astype(np.int32))).to(gpu_device)
    n, L = coords.shape[0], nat.lib()
    assert L.fgx_subm_cache_plan_fits(nat.sz(n), *[C.c_int(d) for d in dims], C.c_int(3), C.c_int(3), C.c_int(3), C.c_int(dil[2]))
    walk, alone = torch.empty(n, dtype=torch.int32, device=gpu_device), torch.empty(n, dtype=torch.int32, device=gpu_device)
    plan = torch.full((L.fgx_narrow_plan_bytes(nat.sz(n), C.c_int(27)),), 0xAB, dtype=torch.uint8, device=gpu_device)
    got, want = _build(coords, dims, dil, walk, plan), _build(coords, dims, dil, alone, None)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and torch.equal(walk, alone)
    nmap, rows_of, raw = got[0].cpu().numpy().view(np.uint32), walk.cpu().numpy().view(np.uint32), plan.cpu().numpy()
    chunks, overflowing, most = -(-n // ROWS), 0, 0
    stride = (len(raw) - HEADER) // chunks
    for c in range(chunks):
        one = raw[HEADER + c * stride:HEADER + (c + 1) * stride]
        table = one[:ROWS * STRIDE * 2].view(np.uint16).reshape(ROWS, STRIDE).astype(np.int64)
        sources = one[ROWS * STRIDE * 2:ROWS * STRIDE * 2 + SLOTS * 4].view(np.uint32)
        rows = one[ROWS * STRIDE * 2 + SLOTS * 4:ROWS * STRIDE * 2 + SLOTS * 4 + ROWS * 4].view(np.uint32)
        here = rows_of[c * ROWS:(c + 1) * ROWS]
        assert np.array_equal(rows[:len(here)], here) and (rows[len(here):] == 0xFFFFFFFF).all()
        entries = np.full((ROWS, 27), 0xFFFFFFFF, np.uint32)
        entries[:len(here)] = nmap[here]
        lost, slot = table[:, :27] == 0xFFFF, table[:, :27] >> 6
        assert (slot[entries == 0xFFFFFFFF] == SLOTS).all() and (table[:, 27:31] == SLOTS * 64).all()
        held = (entries != 0xFFFFFFFF) & ~lost
        assert np.array_equal(sources[slot[held]], entries[held]) and ((table[:, :27][held] >> 4) & 3 == (slot[held] >> 2) & 3).all()
        assert np.array_equal(table[:, STRIDE - 1] != 0, lost.any(1))
        # (a chunk's own rows are held first, whether or not they are anybody's neighbor)
        distinct = len(np.unique(np.concatenate([entries[entries != 0xFFFFFFFF], here])))
        room = SLOTS - (ROWS - len(here))
        assert lost.any() == (distinct > room)
        if distinct <= 1024:                                # (all of them found a place in the builder's table)
            assert len(np.unique(np.concatenate([entries[held], here]))) == min(distinct, room)
        overflowing += bool(lost.any())
        most = max(most, distinct)
    assert (overflowing > 0) == solid and (most > 1024 or dil != (4, 5, 7))
    assert raw[:4].view(np.uint32)[0] == overflowing and not raw[4:HEADER].any()


def test_plan_needs_a_walk_and_a_cube():
    L = nat.lib()
    fits = lambda n, dims, k, d: bool(L.fgx_subm_cache_plan_fits(nat.sz(n), *[C.c_int(x) for x in dims], *[C.c_int(x) for x in k], C.c_int(d)))
    assert fits(100, (1, 204, 204, 204), (3, 3, 3), 16)
    assert not fits(100, (1, 100, 100, 100), (3, 3, 3), 1)              # the form without a walk
    assert not fits(100, (1, 204, 204, 204), (3, 3, 1), 1) and not fits(100, (1, 204, 204, 204), (3, 3, 3), 17) and not fits(0, (1, 204, 204, 204), (3, 3, 3), 1)
