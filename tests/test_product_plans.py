"""Which kernel a product takes, by the rules of the launchers: they look at sizes alone, so they are asked here without a GPU."""
import ctypes

import pytest

MODES = {"store": 0, "add": 1, "gated": 2}


@pytest.fixture(scope="module")
def lib():
    from xeno_rt_amd.ops import build
    return ctypes.CDLL(build.find_library() or build.build())


# w goes past the caches only where it cannot stay in the last one (256 MB) until the next step: a gated matrix of more than two thirds of that, the matrix back from a
# feed-forward of 16384 or wider of more than a third; and only where one row of tiles reads it.
@pytest.mark.parametrize("m,n,k,mode,past", [
    (17, 3072, 1024, "gated", 0), (64, 8192, 2048, "gated", 0), (40, 14336, 4096, "gated", 1), (64, 10922, 4096, "gated", 0), (64, 10928, 4096, "gated", 1),
    (72, 8192, 2048, "gated", 0), (128, 3072, 1024, "gated", 0), (100, 14336, 4096, "gated", 1), (128, 8192, 2048, "gated", 0),
    (129, 14336, 4096, "gated", 0), (200, 8192, 2048, "gated", 0), (256, 6144, 8192, "gated", 0),
    (24, 2048, 2048, "add", 0), (64, 2048, 8192, "add", 0), (20, 256, 16448, "add", 0), (32, 5120, 25600, "add", 1), (64, 2048, 25600, "add", 1), (64, 1024, 25600, "add", 0), (45, 1792, 16384, "gated", 0), (45, 2816, 16384, "gated", 1),
    (40, 4096, 14336, "add", 0), (65, 5120, 25600, "add", 0), (64, 131072, 2048, "store", 1), (64, 32000, 2048, "store", 0)])
def test_w_goes_past_the_caches_only_where_it_cannot_stay_there(lib, m, n, k, mode, past):
    assert lib.xrt_linear_past_caches(m, n, k, MODES[mode]) == past


# Gated products of 17 to 64 rows: in one round of tiles of 64 rows of w, unsplit, where k is short for the number of tiles; in parts along k where a few workgroups would
# walk all of a long k alone.
@pytest.mark.parametrize("m,n,k,unsplit", [
    (17, 40, 128, True), (33, 8192, 192, True), (24, 3072, 1024, True), (64, 8192, 2048, True), (64, 8192, 4160, True), (64, 32, 512, True), (17, 512, 768, True),
    (64, 5120, 3072, False), (64, 704, 4096, False), (64, 1000, 5248, False), (30, 1408, 2048, False), (25, 688, 16320, False), (48, 72, 2048, False), (17, 64, 6400, False), (64, 2816, 4096, False)])
def test_gated_products_of_few_rows_walk_a_long_k_in_parts(lib, m, n, k, unsplit):
    rows, columns = ctypes.c_int(), ctypes.c_int()
    parts = lib.xrt_linear_parts(m, n, k, MODES["gated"], 0, ctypes.byref(rows), ctypes.byref(columns))
    assert (parts, columns.value) == (1, 64) if unsplit else parts >= 3 and columns.value == 128


# Float32 products of a short k, which are little but a tile's start and end: not in many small tiles, nor in large ones where results leave one by one; six blocks where five make two
# rounds and seven leave compute units without work.
@pytest.mark.parametrize("m,n,k,mode,tile", [
    (358, 3536, 8, "gated", 96), (1479, 844, 8, "gated", 96), (223, 5756, 40, "gated", 112), (551, 2484, 192, "gated", 96), (354, 3272, 348, "gated", 96), (886, 948, 16, "gated", 32),
    (281, 1890, 60, "add", 16), (1149, 478, 4, "add", 16), (1699, 1328, 4, "gated", 80), (17, 64, 100, "store", 16), (777, 2048, 2048, "add", 112)])
def test_float32_products_of_a_short_k_take_the_tile_that_ends_soonest(lib, m, n, k, mode, tile):
    rows, together = ctypes.c_int(), ctypes.c_int()
    assert lib.xrt_linear_float_tile(m, n, k, MODES[mode], ctypes.byref(rows), ctypes.byref(together)) == 0
    assert rows.value == tile


# Products that are not gated, more than 64 rows: uncut where two parts take longer (the ends of an adding product's tiles are cheaper than a second kernel when k is short), and
# by the rule for tiles of 128 and 256 rows where there are more rows of x or of w than the finer estimate was fitted to.
@pytest.mark.parametrize("m,n,k,mode,parts", [
    (300, 4096, 256, "add", 1), (597, 1536, 256, "add", 1), (863, 1344, 512, "add", 1), (96, 10240, 256, "add", 1), (788, 2048, 768, "add", 1), (152, 5248, 128, "add", 1), (188, 2288, 256, "add", 2), (241, 1040, 24320, "store", 7),
    (74, 25600, 1024, "add", 1), (79, 28672, 768, "add", 1), (5300, 1024, 3072, "add", 1), (3763, 256, 7168, "add", 4), (3522, 256, 3072, "store", 2), (2932, 128, 2496, "store", 3),
    (2600, 2048, 8192, "add", 2), (4300, 1024, 3072, "add", 2), (4700, 1024, 2624, "add", 1), (100, 2048, 2048, "add", 4), (333, 4096, 14336, "add", 8)])
def test_products_that_are_cut_along_k_and_those_that_are_not(lib, m, n, k, mode, parts):
    rows, columns = ctypes.c_int(), ctypes.c_int()
    assert lib.xrt_linear_parts(m, n, k, MODES[mode], 0, ctypes.byref(rows), ctypes.byref(columns)) == parts


# Every tile of every part is taken by one workgroup and no other, whichever way they are dealt to the eight dies (workgroup i runs on die i % 8); by parts, no die has more than
# its share. By parts: tiles of 256 rows of w from k = 2112 on, narrower ones from k = 6208 on, and any that make a round less so; narrower ones not where the rows of tiles are many,
# except in 8 parts.
@pytest.mark.parametrize("m,n,k,mode,by_parts", [
    (40, 4096, 4096, "add", 0), (61, 4096, 14336, "add", 1), (24, 2816, 2048, "store", 1), (64, 1000, 5248, "gated", 0), (100, 2048, 2048, "add", 0), (65, 3072, 1024, "store", 0),
    (333, 4096, 14336, "add", 1), (333, 4096, 4096, "add", 0), (257, 2048, 14336, "store", 1), (778, 2048, 8192, "store", 1), (300, 12320, 2048, "add", 0), (150, 2664, 5504, "add", 1), (241, 1040, 24320, "store", 1), (520, 2048, 8192, "store", 1), (1100, 4096, 8192, "store", 1),
    (199, 8200, 4096, "store", 1), (333, 6144, 4096, "store", 0), (700, 1000, 8192, "gated", 1), (2000, 1024, 3072, "add", 0),
    (4998, 336, 11904, "gated", 0), (4548, 144, 14976, "gated", 0), (2300, 64, 9024, "gated", 0), (1838, 88, 7040, "store", 1), (2450, 96, 15168, "gated", 1)])
def test_every_tile_of_every_part_has_one_workgroup(lib, m, n, k, mode, by_parts):
    rows, columns, dealt = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    parts = lib.xrt_linear_parts(m, n, k, MODES[mode], 0, ctypes.byref(rows), ctypes.byref(columns))
    groups = lib.xrt_linear_part_order(m, n, k, MODES[mode], 0, ctypes.byref(dealt), None, 0)
    places = (ctypes.c_int * groups)()
    assert lib.xrt_linear_part_order(m, n, k, MODES[mode], 0, ctypes.byref(dealt), places, groups) == groups
    assert dealt.value == by_parts
    tiles = -(-m // rows.value) * -(-(2 * n if mode == "gated" else n) // columns.value)
    assert sorted(place for place in places if place >= 0) == list(range(parts * tiles))
    if by_parts:
        assert groups < parts * tiles + 8
        assert max(sum(place >= 0 for place in places[die::8]) for die in range(8)) == -(-parts * tiles // 8)


# The same of products that are not cut. Side by side on a die (workgroups i, i + 8, ..): tiles of one column where there are up to four rows of them, of one row in panels of
# eight otherwise, and wherever k is no multiple of 64.
@pytest.mark.parametrize("tiles_m,tiles_n,k,down", [(3, 96, 4096, True), (3, 96, 4128, False), (4, 50, 64, True), (4, 50, 72, False), (5, 40, 4096, False), (1, 300, 4100, True),
                                                    (2, 7, 320, True), (40, 6, 2048, False), (9, 13, 100, False)])
def test_every_tile_has_one_workgroup(lib, tiles_m, tiles_n, k, down):
    groups = lib.xrt_linear_tile_order(tiles_m, tiles_n, k, None, 0)
    places = (ctypes.c_int * groups)()
    assert lib.xrt_linear_tile_order(tiles_m, tiles_n, k, places, groups) == groups
    assert groups < tiles_m * tiles_n + 8 and sorted(place for place in places if place >= 0) == list(range(tiles_m * tiles_n))
    first, second = places[0], places[8]
    assert second - first == (1 if tiles_m == 1 or not down else tiles_n)


# 17 to 64 rows, not gated: at most one workgroup to a compute unit, and fewer parts than that leaves room for where their sums cost more than they save.
@pytest.mark.parametrize("m,n,k,parts", [(20, 12288, 8192, 2), (28, 9104, 16448, 3), (20, 12496, 7680, 2), (32, 12288, 14336, 2), (61, 4096, 1024, 4), (64, 3072, 2048, 4), (64, 3008, 1024, 4),
                                         (61, 4096, 14336, 8), (40, 16384, 2048, 2), (40, 16512, 2048, 1)])
def test_few_rows_take_no_more_than_a_workgroup_a_compute_unit(lib, m, n, k, parts):
    rows, columns = ctypes.c_int(), ctypes.c_int()
    assert lib.xrt_linear_parts(m, n, k, MODES["add"], 0, ctypes.byref(rows), ctypes.byref(columns)) == parts
    assert parts * -(-n // columns.value) <= 256
