"""Segment tables of the row tiles and the streaming GEMM's item order, at the numbers of tiles where their kernels change."""
import ctypes as C

import numpy as np
import pytest
import torch

from flexgemm_amd import _native as nat

pytestmark = pytest.mark.gpu


def _codes(n, seed, bits=27):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 1 << bits, n, dtype=np.int64) & rng.integers(0, 1 << bits, n, dtype=np.int64)
    codes[rng.random(n) < 0.1] = 0
    return codes.astype(np.int32)


# one tile, one turn of the single workgroup and one more tile, its last number of tiles and the first in chunks, a chunk's first and last
# tile, more chunks than the workgroup that adds them up has threads
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 8191, 8192, 8193, 12287, 12288, 12289, 83350, 2667120, 4 * 1024 * 1024 + 4097])
@pytest.mark.parametrize("which", ["both", "seg", "plan"])
def test_segment_tables(gpu_device, n, which):
    print(f"[case] tile segment tables n={n} {which}", flush=True)
    codes = _codes(n, n)
    dev = torch.from_numpy(codes).to(gpu_device)
    count = np.array([bin(c).count("1") for c in range(1 << 14)], np.int64)
    pop = count[codes & 0x3FFF] + count[(codes >> 14) & 0x3FFF]
    seg, plan = [torch.full((n + 2,), -7, dtype=torch.int32, device=gpu_device) for _ in range(2)]
    nat.check(nat.lib().fgx_tile_plan(None, None, None, nat.sz(n), C.c_int(1), C.c_int(1), C.c_int(1), nat.ptr(dev),
                                      nat.ptr(seg) if which != "plan" else None, nat.ptr(plan) if which != "seg" else None, None, None, C.c_int(1),
                                      C.c_int(1), C.c_int(1), None, None, nat.stream()))
    for got, per_tile, made in ((seg, pop, which != "plan"), (plan, np.maximum(pop, 1), which != "seg")):
        want = np.concatenate([[0], np.cumsum(per_tile), [-7]]) if made else np.full(n + 2, -7)
        assert np.array_equal(got.cpu().numpy(), want)


def test_plan_count_of_very_many_tiles(gpu_device):
    n = (1 << 26) + 5
    print(f"[case] plan count of {n} tiles", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(1)
    codes = torch.randint(0, 8, (n,), generator=gen, device=gpu_device, dtype=torch.int32)
    seg = torch.empty(n + 1, dtype=torch.int32, device=gpu_device)
    L = nat.lib()
    ws = nat.workspace(L.fgx_tile_workspace_bytes(nat.sz(n), C.c_int(1)), gpu_device)
    nat.check(L.fgx_gather_plan_count(nat.ptr(codes), nat.sz(n), nat.ptr(seg), nat.ptr(ws), nat.sz(ws.numel()), nat.stream()))
    pop = ((codes & 1) + (codes >> 1 & 1) + (codes >> 2)).clamp_(min=1).cumsum(0)
    assert int(seg[0]) == 0 and torch.equal(seg[1:], pop.to(torch.int32))


def _dealt(cost_bin, slabs, groups):
    """The order of fgx_gather_item_order: items by cost, round after round to the least loaded slot first, the cheapest in the round
    that is not full."""
    total = len(cost_bin)
    by_cost = np.argsort(cost_bin, kind="stable").astype(np.int64)
    rounds, rem = divmod(total, groups)
    scale = 0
    while ((rounds + 1) * (32 * slabs + 3)) >> scale >= 1 << 21:
        scale += 1
    cost = (np.maximum(32 - cost_bin, 1) * slabs + 3) >> scale
    out, load = np.empty(total, np.int64), np.arange(groups, dtype=np.int64)
    if rem:
        out[rounds * groups:] = by_cost[total - rem:]
        load[:rem] += cost[by_cost[total - rem:]] << 10
    for r in range(rounds):
        slots = np.argsort(load)
        items = by_cost[r * groups:(r + 1) * groups]
        out[r * groups + slots] = items
        load[slots] += cost[items] << 10
    return out


# few items and slots; past the list kept in LDS; past the 26 bits that hold an item beside its cost
@pytest.mark.parametrize("tiles,col_tiles,groups,slabs", [(5, 1, 3, 1), (1306, 1, 256, 2), (9001, 3, 500, 4), ((1 << 25) + 3, 2, 1024, 1)])
def test_item_order(gpu_device, tiles, col_tiles, groups, slabs):
    print(f"[case] item order of {tiles} x {col_tiles} items in {groups} slots", flush=True)
    codes = _codes(tiles, tiles)
    dev = torch.from_numpy(codes).to(gpu_device)
    total = tiles * col_tiles
    item_at = torch.full((total,), -1, dtype=torch.int32, device=gpu_device)
    L = nat.lib()
    ws = nat.workspace(L.fgx_gather_item_order_workspace_bytes(nat.sz(tiles), C.c_int(col_tiles)), gpu_device)
    nat.check(L.fgx_gather_item_order(nat.ptr(dev), nat.sz(tiles), C.c_int(col_tiles), C.c_int(slabs), C.c_int(groups), nat.ptr(ws),
                                      nat.sz(ws.numel()), nat.ptr(item_at), nat.stream()))
    got = item_at.cpu().numpy()
    count = np.array([bin(c).count("1") for c in range(1 << 14)], np.int64)
    cost_bin = 32 - np.repeat(count[codes & 0x3FFF] + count[(codes >> 14) & 0x3FFF], col_tiles)
    assert np.array_equal(got, _dealt(cost_bin, slabs, groups))
