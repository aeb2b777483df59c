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


@pytest.mark.parametrize("groups,top,N,K", [(64, 6, 512, 1024), (128, 8, 768, 2048), (32, 4, 1536, 2048), (17, 2, 4096, 1536)])
def test_many_groups_of_few_entries_take_the_first_five_tiles(groups, top, N, K):
    """Beyond sixteen groups, below 200 entries a group: none of the tiles that are for many steps of few groups; at sixteen, and from 200 on, some."""
    pick = hip_ops.library("experts").cdll.tis_grouped_tile
    few = {pick(1, groups, rows, c_long(rows * top), N, K, 0) for rows in range(17, 200 * groups // top, 7)}
    assert few <= {-1, 0, 1, 2, 3, 4}
    more = {pick(1, g, rows, c_long(rows * top), N, K, 0) for g in (16, groups) for rows in range(-(-200 * g // top), 4000 * g // top, 41)}
    assert more & {6, 7, 8}


@pytest.mark.parametrize("rows,N,K,tile", [(3000, 2816, 1024, 3), (3492, 15104, 384, 3), (7321, 9088, 704, 3), (1531, 48000, 1536, 0),
                                           (300, 448, 512, 6)])
def test_many_results_of_few_steps(rows, N, K, tile):
    """Products whose results take a good part of their time: the tiles (0: 256 x 256, 3: 128 x 192 two a unit, 6: 64 x 64) that were measured to be the
    fastest, each by a twentieth to a quarter against the tile that an estimate by the steps alone picks."""
    assert hip_ops.library("gemm_tiles").cdll.tis_gemm_tiles_pick(rows, N, K) == tile


@pytest.mark.parametrize("groups,top,rows,N,K,split", [
    # slower with the sum over K split, by 4 to 24 %
    (128, 8, 1, 5632, 384, False), (128, 8, 1, 5632, 512, False), (16, 4, 16, 2048, 384, False), (16, 4, 16, 2048, 512, False), (16, 4, 16, 2048, 704, False),
    (32, 4, 16, 1024, 512, False), (64, 8, 40, 512, 704, False), (8, 2, 16, 5632, 704, False), (64, 8, 5, 2048, 384, False),
    # faster, by 4 to 100 %
    (8, 2, 1, 2048, 2816, True), (8, 2, 8, 5632, 2048, True), (16, 4, 16, 5632, 2048, True), (64, 8, 16, 2048, 2048, True), (128, 8, 8, 2048, 1536, True),
    (64, 8, 5, 1024, 1024, True), (8, 2, 5, 2816, 1024, True), (8, 2, 5, 1024, 1408, True), (64, 8, 5, 512, 384, True), (16, 4, 16, 1024, 704, True), (8, 2, 1, 2048, 384, True)])
def test_sums_over_k_are_split_where_that_was_faster(groups, top, rows, N, K, split):
    """A sum over K goes to a workgroup's four waves from 1,536 terms on, and below while the blocks of columns are few."""
    lib = hip_ops.library("experts").cdll
    assert lib.tis_grouped_tile(1, groups, rows, c_long(rows * top), N, K, 0) < 0
    assert bool(lib.tis_grouped_split(1, groups, rows, c_long(rows * top), N, K)) == split


@pytest.mark.parametrize("heads,rows,N,K,split", [
    # a product per head; slower with the sum over K split, by 5 to 25 %
    (64, 32, 128, 1024, False), (128, 16, 128, 512, False), (32, 63, 128, 1536, False), (64, 63, 64, 512, False), (128, 16, 512, 1536, False), (128, 32, 128, 1024, False),
    (80, 16, 192, 1024, False), (112, 32, 128, 512, False),
    # faster
    (16, 16, 128, 512, True), (64, 5, 128, 512, True), (32, 1, 128, 1536, True), (64, 16, 192, 512, True), (64, 32, 64, 512, True), (64, 32, 192, 512, True), (128, 1, 192, 512, True)])
def test_products_per_head_are_split_where_that_takes_fewer_rounds(heads, rows, N, K, split):
    assert bool(hip_ops.library("experts").cdll.tis_grouped_split(0, heads, rows, c_long(rows), N, K)) == split


@pytest.mark.parametrize("rows,D,F,H,G,HD,keys,takes", [
    # slower in one kernel, by 5 to 45 %
    (1, 64, 192, 2, 1, 32, 512, False), (64, 64, 192, 2, 1, 32, 512, False), (1, 64, 176, 2, 1, 24, 384, False), (1, 64, 128, 1, 1, 40, 192, False), (260, 32, 96, 4, 4, 8, 384, False),
    (320, 60, 176, 5, 1, 12, 384, False), (260, 64, 176, 2, 1, 24, 192, False), (512, 64, 192, 2, 1, 32, 512, False), (260, 64, 128, 1, 1, 40, 64, False), (260, 32, 88, 2, 1, 16, 256, False),
    (300, 64, 192, 4, 2, 16, 512, False),
    # faster, or as fast
    (1, 64, 176, 8, 2, 8, 512, True), (256, 64, 176, 8, 4, 8, 512, True), (512, 64, 176, 8, 2, 8, 512, True), (1, 64, 192, 2, 1, 32, 256, True), (256, 64, 192, 4, 2, 16, 512, True),
    (1, 64, 128, 1, 1, 40, 128, True), (260, 32, 96, 4, 4, 8, 256, True), (320, 64, 192, 16, 4, 4, 512, True), (512, 60, 176, 5, 1, 12, 192, True)])
def test_small_blocks_where_one_kernel_was_faster(rows, D, F, H, G, HD, keys, takes):
    assert bool(hip_ops.library("small_block").cdll.tis_small_block_takes(rows, D, F, H, G, HD, keys, 16)) == takes
