"""The plans of prompts' products are kept by 64 and 128 rows: what they are made of changes at those lines alone, and a length that is not seen for the first time
within them asks for no search."""

import ctypes
import random

import pytest

from flyweight_amd.kernels import ops


@pytest.fixture(scope="module", autouse=True)
def library():
    ops.library()


def shapes(count, seed):
    rng = random.Random(seed)
    for _ in range(count):
        yield rng.randrange(3), int(2 ** rng.uniform(6.03, 12.5)), int(2 ** rng.uniform(4, 14)), 32 * int(2 ** rng.uniform(0, 9))


def test_the_tiles_rows_are_multiples_of_64():
    for table in (*ops._TIME_LARGE.values(), *ops._TIME_LARGE_CUT.values()):
        assert all(tile[0] % 64 == 0 for tile in table)


def test_the_estimates_are_of_every_tile_there_is():
    """The tables' tiles and the kernels' are the same, K cut on those that have it (and on 128 x 256, which a rule of its own chooses)."""
    have = ctypes.c_size_t(0), ctypes.c_int(0)
    for mode in range(3):
        takes = lambda tile, slices: ops.library().fw_gemm_mfma_big_tile_needs(mode, 1000, 1000, 4096, *tile, slices, *map(ctypes.byref, have)) == 0    # noqa: E731
        tiles = [(rows, columns, each) for rows in range(32, 353, 32) for columns in range(32, 417, 32) for each in (1, 2, 3)]
        assert {tile for tile in tiles if takes(tile, 1)} == set(ops._TIME_LARGE[mode])
        cut = {(rows, columns, 1) for rows, columns in ops._TIME_LARGE_CUT.get(mode, {})}
        assert {tile for tile in tiles if takes(tile, 2)} == (cut | {(128, 256, 1)} if cut else set())


def test_what_the_plans_are_made_of_changes_at_their_lines_alone():
    def needs(mode, M, N, K, tile):
        have = ctypes.c_size_t(0), ctypes.c_int(0)
        ops._check(ops.library().fw_gemm_mfma_big_tile_needs(mode, M, N, K, *tile, *map(ctypes.byref, have)))
        return tuple(v.value for v in have)

    for mode, M, N, K in shapes(400, 1):
        assert ops._tiled_times(mode, M, N, K) == ops._tiled_times(mode, -(-M // 128) * 128, N, K)
        tile = ops.large_tile(mode, M, N, K)
        if tile is not None:
            assert tile == ops._fastest_large(mode, -(-M // 64), N, K)[0] and tile[4:] == needs(mode, M, N, K, tile[:4])


def test_a_new_length_asks_for_no_search_where_a_neighbour_has():
    lines = (ops._fastest_large, ops._fastest_older)
    for mode, M, N, K in shapes(60, 2):
        first = ops.ROWS_MAX + M // 64 * 64 + 1             # beyond the rows of the product whose waves split K
        ops.large_tile(mode, first, N, K)
        before = [line.cache_info().misses for line in lines]
        for rows in range(first + 1, first + 64):
            ops.large_tile(mode, rows, N, K)
        assert [line.cache_info().misses for line in lines] == before
