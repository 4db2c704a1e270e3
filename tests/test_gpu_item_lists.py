"""The weight gradient's balanced work lists: every item on one list, and no workgroup far above the mean, over the builder's sizes."""
import ctypes as C

import numpy as np
import pytest
import torch

from flexgemm_amd import _native as nat

pytestmark = pytest.mark.gpu


# one chunk an XCD and fewer; chunks dealt one by one and beyond; fewer items than a batch on an XCD; more than 32 tiles (several chunks a unit); most items
@pytest.mark.parametrize("nb,v,tiles", [(1, 3, (1, 1)), (2, 8, (1, 2)), (1, 27, (1, 2)), (3, 27, (1, 1)), (12, 27, (1, 1)), (16, 27, (3, 3)), (5, 27, (5, 6)), (2, 27, (5, 7)), (1, 27, (8, 13))])
@pytest.mark.parametrize("empty", [0.0, 0.3])
def test_lists(nb, v, tiles, empty):
    L, rows = nat.lib(), 4096
    n, co, ci = nb * rows, tiles[0] * 128, tiles[1] * 128
    rng = np.random.default_rng(nb + v)
    pairs = (rng.random((v, nb)) ** 2 * rows * (rng.random((v, nb)) >= empty)).astype(np.int64)
    pairs[v // 2] = rows
    bounds = np.concatenate([np.zeros((v, 1), np.int64), np.cumsum(pairs, 1)], 1)
    bounds += np.concatenate([[0], np.cumsum(bounds[:-1, -1])])[:, None]
    dev = torch.from_numpy(bounds.astype(np.int32)).cuda()
    args = (nat.sz(n), C.c_int(v), C.c_int(ci), C.c_int(co), C.c_int(128), C.c_int(128), C.c_int(rows))
    words = L.fgx_wgrad_item_lists_count(*args)
    assert words > 0
    out = torch.full((words + 1,), -7, dtype=torch.int32, device="cuda")
    nat.check(L.fgx_wgrad_item_lists(nat.ptr(dev), *args, nat.ptr(out), nat.stream()))
    w = out.cpu().numpy().view(np.uint32).astype(np.int64)
    groups, items, per = int(w[0]), int(w[1]), int(w[2])
    assert items == nb * v * per and per == tiles[0] * tiles[1] and w[-1] == 0xFFFFFFF9
    head, nxt = w[4:4 + groups], w[4 + groups:4 + groups + items]
    cost = np.repeat(pairs.T.reshape(-1), per)                      # an item is (block, offset, tile)
    cost = np.where(cost > 0, cost + 1280, 0)                       # (and the builder's fixed share of one that has pairs)
    seen, load = np.zeros(items, bool), np.zeros(groups)
    for g, h in enumerate(head):
        while h != 0xFFFFFFFF:
            assert 0 <= h < items and not seen[h]
            seen[h] = True
            load[g] += cost[h]
            h = nxt[h]
    assert seen.all()
    # an XCD takes whole chunks (at most 32 tiles of a unit) to within one of them, a workgroup whole items to within two
    chunk = cost.max() * min(per, 32) * 8 / groups
    assert load.max() <= cost.sum() / groups + chunk + 2 * cost.max()


@pytest.mark.parametrize("n,rows", [(131071, 44032), (131072, 22528), (393216, 24576), (393217, 30720), (524288, 32768), (600000, 60416)])
def test_blocks_of_nine_tiles(n, rows):
    s = nat.table_lookup(nat.PASS_WGRAD, torch.bfloat16, n, 272, 384, 27)
    assert (s.tile_rows, s.tile_cols, s.stream, s.block_rows) == (128, 128, 1, rows)
