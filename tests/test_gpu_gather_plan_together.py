"""Gather plans whose short tiles are filled two and four to a workgroup: around the counts of tiles where that starts, and with every remainder."""
import pytest

import test_gpu_gather_plan as one_by_one

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,tile_rows", [(511, 64), (512, 64), (513, 64), (1023, 64), (1024, 64), (1025, 64), (1026, 64), (1027, 64), (511, 128), (512, 128), (513, 128),
                                             (600, 192), (600, 256)])
@pytest.mark.parametrize("short", [0, 63])
def test_plan(tiles, tile_rows, short):
    for v, col_tiles in ((27, 1), (8, 0)):
        one_by_one.test_plan_against_numpy(tiles * tile_rows - short, tile_rows, v, col_tiles)
