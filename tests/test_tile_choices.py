"""Which tile a product takes: the estimates behind the choice, asked on the host."""
from __future__ import annotations

from ctypes import c_long

import pytest

from tiny_inference_server_amd.ops import hip_ops

GROUPED_ROWS = (128, 64, 128, 256, 128, 64, 128, 256, 192)     # rows of the grouped product's tiles, in the order of its choice


@pytest.mark.parametrize("groups,top,N,K", [(64, 8, 1024, 1408), (64, 6, 512, 1024), (32, 2, 2048, 704), (128, 8, 2048, 768), (8, 2, 2816, 1024), (4, 1, 1024, 2048)])
def test_groups_of_few_entries_take_no_high_tiles(groups, top, N, K):
    """However many groups there are, a tile of more than 128 rows has groups that fill three quarters of one on average."""
    pick = hip_ops.library("experts").cdll.tis_grouped_tile
    high = 0
    for rows in list(range(1, 1200, 13)) + [1531, 2048, 3000, 6000, 20000]:
        tile = pick(1, groups, rows, c_long(rows * top), N, K, 0)
        if tile >= 0 and GROUPED_ROWS[tile] > 128:
            assert 4 * rows * top >= 3 * groups * GROUPED_ROWS[tile], (rows, tile)
            high += 1
    assert high
