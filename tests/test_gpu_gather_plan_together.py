"""Gather plans whose short tiles are filled two and four to a workgroup: around the counts of tiles where that starts, and with every remainder."""
import ctypes as C

import pytest
import torch

from flexgemm_amd import _native as nat
import test_gpu_gather_plan as one_by_one

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,tile_rows", [(511, 64), (512, 64), (513, 64), (1023, 64), (1024, 64), (1025, 64), (1026, 64), (1027, 64), (511, 128), (512, 128), (513, 128),
                                             (600, 192), (600, 256)])
@pytest.mark.parametrize("short", [0, 63])
def test_plan(tiles, tile_rows, short):
    for v, col_tiles in ((27, 1), (8, 0)):
        one_by_one.test_plan_against_numpy(tiles * tile_rows - short, tile_rows, v, col_tiles)


# items of the plan's own workgroup of 512 threads against the launch of its own (1 024 threads): the fewest slots that are sorted, all of a workgroup's, a round
# that is not full
@pytest.mark.parametrize("groups", [256, 257, 511, 512])
@pytest.mark.parametrize("tiles,col_tiles", [(300, 2), (512, 2), (1500, 1), (1500, 3)])
def test_item_order_beside_the_plan(groups, tiles, col_tiles):
    n, v, L = tiles * 64, 27, nat.lib()
    g = torch.Generator().manual_seed(tiles)
    nmap = torch.randint(0, n, (n, v), generator=g, dtype=torch.int32)
    nmap[torch.rand(n, v, generator=g) < torch.rand(n, 1, generator=g) ** 0.02] = -1
    gray = ((nmap >= 0).long() << torch.arange(v)).sum(1).int().cuda()
    nmap, order = nmap.cuda(), torch.arange(n).cuda()
    code, seg = torch.empty(tiles, dtype=torch.int32, device="cuda"), torch.empty(tiles + 1, dtype=torch.int32, device="cuda")
    idx, band = torch.empty(tiles * v, 64, dtype=torch.int32, device="cuda"), torch.empty(tiles * v, dtype=torch.int32, device="cuda")
    beside, alone = (torch.full((tiles * col_tiles,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    ws = nat.workspace(L.fgx_gather_item_order_workspace_bytes(nat.sz(tiles), C.c_int(col_tiles)), torch.device("cuda"))
    nat.check(L.fgx_tile_plan(nat.ptr(gray), nat.ptr(order), nat.ptr(nmap), nat.sz(n), C.c_int(v), C.c_int(64), C.c_int(0), nat.ptr(code), None, nat.ptr(seg),
                              nat.ptr(idx), nat.ptr(band), C.c_int(col_tiles), C.c_int(2), C.c_int(groups), nat.ptr(ws), nat.ptr(beside), nat.stream()))
    nat.check(L.fgx_gather_item_order(nat.ptr(code), nat.sz(tiles), C.c_int(col_tiles), C.c_int(2), C.c_int(groups), nat.ptr(ws), nat.sz(ws.numel()),
                                      nat.ptr(alone), nat.stream()))
    assert torch.equal(beside, alone) and torch.equal(beside.sort().values, torch.arange(tiles * col_tiles, dtype=torch.int32, device="cuda"))
