"""Launch plans at the limits of a launch: work items along an axis fit 32 bits, so a launch of 256-thread workgroups
holds fewer than 2^24 of them."""
import random

import numpy as np
import pytest

import host_plans as P

MOST_BLOCKS = (2**32 - 1) // 256


@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_direct_tiles_fit_the_launch(dtype):
    # 33 x 17 pixels take four tiles: the last batch that fits, and the first that does not
    assert P.direct_tiles(dtype, MOST_BLOCKS // 4, 1, 301, 211, 17, 33)[0] == MOST_BLOCKS // 4 * 4
    assert P.direct_tiles(dtype, MOST_BLOCKS // 4 + 1, 1, 301, 211, 17, 33) is None
    # large planes: 724 x 1448 tiles an item; sixteen items fit and seventeen do not
    assert P.direct_tiles(dtype, 16, 1, 301, 211, 23168, 23168)[0] < 2**24
    assert P.direct_tiles(dtype, 17, 1, 301, 211, 23168, 23168) is None
    # a workgroup per CU at least: tiles, or tiles times runs of four channels
    assert P.direct_tiles(dtype, 255, 1, 301, 211, 16, 32) is None
    assert P.direct_tiles(dtype, 256, 1, 301, 211, 16, 32) == (256, 1)
    assert P.direct_tiles(dtype, 4, 253, 301, 211, 16, 32) == (4, 64) and P.direct_tiles(dtype, 4, 252, 301, 211, 16, 32) is None
    # the counts of a batch beyond 32 bits
    assert P.direct_tiles(dtype, 2**31 - 1, 1, 301, 211, 16000, 16000) is None
    rng = random.Random(7)
    for _ in range(2000):
        n, c = (int(2 ** rng.uniform(0, 31)) for _ in range(2))
        h, w = (int(2 ** rng.uniform(1, 15)) for _ in range(2))
        ho, wo = (int(2 ** rng.uniform(0, 15)) for _ in range(2))
        p = P.direct_tiles(dtype, n, c, h, w, ho, wo)
        if p is not None:
            assert 0 < p[0] <= MOST_BLOCKS and p[0] * 512 >= n * ho * wo and 0 < p[1] <= 65535


@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_resize_gradient_planes_fit_the_launch(dtype):
    # growth by four: tiles of 64 columns by eight rows fill a launch at 2^27 rows
    rows = 8 * (MOST_BLOCKS // 8 * 8)
    assert P.resize_grad_planes(dtype, 1, (rows, 64), (4 * rows, 256)) == (8, MOST_BLOCKS // 8 * 8, 1)
    assert P.resize_grad_planes(dtype, 1, (rows + 1, 64), (4 * rows + 4, 256)) is None
    # planes of one column
    assert P.resize_grad_planes(dtype, 1, (2**31 - 2, 1), (2**31 - 1, 1)) is None
    rng = random.Random(8)
    for _ in range(2000):
        h, w = (int(2 ** rng.uniform(0, 30)) for _ in range(2))
        large = [max(1, int(v * 2 ** rng.uniform(-1, 2))) for v in (h, w)]
        p = P.resize_grad_planes(dtype, int(2 ** rng.uniform(0, 12)), (h, w), large, rng.random() < 0.5)
        if p is not None:
            assert p[0] in (8, 16) and 0 < p[1] <= MOST_BLOCKS and p[1] % 8 == 0 and p[2] > 0


# (type, mode, input, points per item, microseconds by elections and by sorting): measured, grids turned or scattered
GRADIENTS = [
    # pictures and feature maps
    ("fp32", 0, (8, 3, 479, 637), 479 * 637, 2493, 220), ("fp32", 0, (7, 4, 341, 510), 341 * 510, 2127, 133),
    ("fp32", 0, (1, 3, 64, 64), 9 * 256, 32, 22), ("fp32", 0, (1, 3, 64, 64), 64 * 256, 126, 23),
    ("fp32", 2, (1, 3, 64, 64), 3 * 256, 50, 41), ("fp32", 2, (1, 3, 64, 64), 9 * 256, 135, 45),
    # few tap passes
    ("fp32", 0, (1, 3, 64, 64), 4 * 256, 17, 20), ("fp32", 1, (1, 3, 64, 64), 9 * 256, 13, 19),
    ("fp32", 2, (1, 3, 64, 64), 256, 24, 36),
    # large batches, few points on large planes, many on small ones
    ("fp32", 0, (512, 3, 64, 64), 1600, 24.9, 75.6), ("fp16", 0, (1000, 3, 48, 48), 2304, 74.7, 132.9),
    ("fp32", 0, (1, 3, 1080, 1920), 1600, 18.3, 57.6), ("fp16", 0, (8, 3, 512, 512), 1600, 20.6, 55.0),
    ("fp32", 0, (1024, 1, 16, 16), 4096, 99.9, 1014), ("fp32", 0, (512, 1, 16, 16), 2304, 52.4, 194),
    ("fp32", 1, (512, 3, 64, 64), 6561, 44.6, 211), ("fp16", 0, (128, 7, 32, 32), 1600, 64.1, 41.9),
    ("fp32", 2, (512, 3, 64, 64), 4096, 340, 1682), ("fp32", 2, (512, 3, 32, 32), 512, 55, 183),
    ("fp16", 2, (1024, 8, 32, 32), 1024, 220, 758)]


@pytest.mark.parametrize("dtype,interp,shape,points,elections,sorting", GRADIENTS)
def test_input_gradient_takes_the_faster_of_two_variants(dtype, interp, shape, points, elections, sorting):
    assert (P.sorting_takes_planes(dtype, interp, shape, points) is not None) == (sorting < elections)


# (planes, small, large, microseconds by the gather and by the planes kernel): measured, 16-bit rows off the word grid
RESIZES = [(131072, (3, 3), (7, 7), 19.4, 142), (16384, (20, 5), (41, 11), 24.9, 136), (64, (500, 3), (1001, 7), 5.1, 19.6),
           (4096, (40, 9), (81, 19), 21.6, 61), (65536, (7, 7), (15, 15), 48.5, 134), (1, (5000, 5), (10001, 11), 4.4, 7.3),
           (16384, (14, 14), (29, 29), 46.4, 72.7), (32768, (13, 13), (27, 27), 79.9, 123),
           (512, (65, 129), (257, 513), 189, 72), (128, (160, 240), (320, 481), 63, 31), (128, (160, 240), (480, 721), 118, 45)]


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("planes,small,large,gather,tiles", RESIZES)
def test_resize_gradient_of_odd_rows_takes_the_faster_of_two_kernels(dtype, planes, small, large, gather, tiles):
    assert (P.resize_grad_planes(dtype, planes, small, large) is not None) == (tiles < gather)


# (type, planes, small, large, microseconds by rows and by the gather): measured in graphs of 64 calls
FEW = [("bf16", 49, (10, 20), (11, 23), 3.9, 2.5), ("bf16", 35, (21, 187), (31, 281), 4.5, 3.9), ("fp16", 83, (8, 36), (6, 29), 3.6, 2.4),
       ("fp16", 570, (11, 13), (16, 19), 4.3, 3.2), ("bf16", 807, (14, 5), (21, 7), 4.3, 3.1), ("fp16", 144, (9, 196), (11, 245), 4.7, 4.0),
       ("fp32", 7, (51, 51), (56, 57), 3.9, 2.9), ("fp16", 125, (14, 70), (28, 140), 4.6, 4.1), ("bf16", 477, (6, 123), (10, 215), 5.4, 6.0),
       ("bf16", 622, (45, 5), (91, 11), 6.1, 5.0), ("bf16", 4, (32, 18), (80, 45), 4.7, 4.1), ("fp16", 25, (127, 137), (76, 83), 4.8, 4.2),
       ("fp32", 3171, (3, 32), (6, 65), 5.9, 6.1), ("fp32", 20, (116, 284), (145, 355), 6.1, 7.2), ("fp16", 55, (61, 69), (152, 172), 5.9, 7.1),
       ("fp32", 1, (45, 190), (180, 760), 6.6, 7.6)]


@pytest.mark.parametrize("dtype,planes,small,large,rows,gather", FEW)
def test_resize_gradient_of_few_elements_takes_the_faster_kernel(dtype, planes, small, large, rows, gather):
    assert P.resize_grad_kernel(dtype, planes, small, large) == ("gather" if gather < rows else "rows")


@pytest.mark.parametrize("align", [False, True])
def test_resize_gradient_rows_hold_what_an_element_visits(align):
    """growth by four and five, where rounding adds a row or column to 2 / scale: the visits of every element, stepped in single
    precision as the kernels do"""
    f, most = np.float32, 0
    assert P.resize_grad_rows("fp32", 4, (100, 100), (496, 496) if align else (500, 500), align) is not None
    for growth in (4, 5):
        for n in range(16, 260, 3):
            large = growth * (n - 1) + 1 if align else growth * n
            scale = f(n - 1) / f(large - 1) if align else f(n) / f(large)
            offset = f(0.0 if align else 0.5)
            i = np.arange(n, dtype=f)
            start = np.clip(np.ceil((i - f(1) + offset) * (f(1) / scale) - offset), 0, large)
            at, visits = (start + offset) * scale - offset, np.zeros(n, int)
            for k in range(16):
                visits += (at < i + f(1)) & (start + k < large) & (visits == k)
                at = at + scale
            most = max(most, visits.max())
    assert most == 11 and most <= P.resize_grad_rows_visits()


# (bytes of a unit, rows, shrunk, align corners, in pairs): microseconds with kept rows / in pairs
SHRUNK = [(12, 720, 384, False, True),    # 51.6 / 45.0
          (6, 720, 480, False, False),    # 33.3 / 39.0
          (6, 2160, 720, False, False),   # 6.8 / 8.9: every row falls on a source row
          (6, 1974, 658, False, False), (4, 1305, 435, False, False), (2, 1932, 644, False, False),  # 22 / 35, 8.3 / 12, 25 / 35
          (12, 7 * 89 + 1, 90, True, False), (12, 7 * 89 + 2, 90, True, True),  # align corners: a factor of 7, and beside it
          (2, 1000, 400, False, True), (6, 1440, 720, False, True), (12, 750, 500, False, True), (12, 700, 500, False, False)]


@pytest.mark.parametrize("unit,rows,shrunk,align,pairs", SHRUNK)
def test_shrinking_rows_take_the_faster_of_two_kernels(unit, rows, shrunk, align, pairs):
    assert P.shrink_in_pairs(unit, rows, shrunk, align) == pairs


# (type, planes, small, large, non-temporal stores, rows in runs): outputs of 26, 103, 135, 270 and 328 MB; fp32 of which input
# and output together are beyond the last-level cache; rows that shrink
FLAT = [("fp32", 512, (56, 56), (112, 112), True, True), ("fp32", 2048, (56, 56), (112, 112), False, True),
        ("bf16", 512, (65, 129), (257, 513), False, True), ("fp32", 512, (65, 129), (257, 513), True, True),
        ("fp16", 4096, (100, 100), (200, 200), True, False), ("fp32", 2048, (100, 100), (200, 200), True, False),
        ("fp32", 5869, (42, 65), (88, 114), True, False), ("fp32", 4273, (56, 71), (112, 113), True, False),
        ("fp16", 11595, (54, 79), (75, 110), False, True), ("fp32", 64, (112, 112), (56, 56), True, False)]


@pytest.mark.parametrize("dtype,planes,small,large,streaming,runs", FLAT)
def test_flat_resize_rows_and_stores(dtype, planes, small, large, streaming, runs):
    assert P.flat_resize(dtype, planes, small, large) == (streaming, runs)


def test_sorting_scratch_holds_a_group_of_items():
    """a batch's scratch is that of as many items as 256 MiB hold, of one at least; items beyond 4 GiB are left alone"""
    cache = 256 << 20
    assert P.gather_groups("fp32", 0, (8, 3, 479, 637), 479 * 637)[0] == 8  # 58 MiB
    for dtype, interp, shape, points, groups in [("fp32", 2, (16, 3, 1080, 1920), 1080 * 1920, 16),
                                                 ("fp32", 0, (64, 3, 720, 1280), 720 * 1280, 6),
                                                 ("fp16", 0, (45, 1, 480, 641), 480 * 641, 2),
                                                 ("fp32", 0, (300, 1, 9, 20, 21), 39 * 32 * 31, 2)]:
        group, words = P.gather_groups(dtype, interp, shape, points)
        assert -(-shape[0] // group) == groups and (group == 1 or group * words * 4 <= cache), (shape, group, words)
    assert P.gather_groups("fp32", 2, (1, 1, 5300, 5300), 5300 * 5300) is not None  # 3.9 GiB
    assert P.gather_groups("fp32", 2, (1, 1, 5800, 5800), 5800 * 5800) is None
    assert P.gather_groups("fp32", 0, (65536, 1, 9, 9), 2000) is None
    rng = random.Random(9)
    for _ in range(2000):
        n, c, h, w = (int(2 ** rng.uniform(0, k)) for k in (16, 10, 13, 13))
        p = P.gather_groups(rng.choice(["fp32", "fp16"]), rng.choice([0, 1, 2]), (n, c, h, w), int(2 ** rng.uniform(8, 25)))
        if p is not None:
            assert 1 <= p[0] <= n and (p[0] == 1 or p[0] * p[1] * 4 <= cache) and p[1] * 4 <= 4 << 30


# (type, mode, padding, input, points per item, microseconds by lists and by tiles): measured
TILES = [("fp32", 0, 0, (8, 3, 479, 637), 479 * 637, 178, 86), ("fp16", 0, 2, (1, 14, 236, 198), 229 * 192, 32, 20),
         ("fp32", 0, 1, (8, 3, 479, 637), 479 * 637, 455, 330), ("fp32", 0, 1, (1, 3, 480, 640), 480 * 640, 73, 110),
         ("fp32", 0, 1, (2, 2, 200, 300), 200 * 300, 51, 101), ("fp32", 0, 0, (21, 60, 40, 40), 77 * 77, 86, 156),
         ("fp16", 0, 0, (10, 2, 267, 440), 448 * 738, 314, 111), ("fp32", 0, 1, (14, 4, 33, 56), 62 * 106, 60, 93),
         ("bf16", 0, 0, (2, 5, 96, 192), 162 * 324, 31, 40), ("bf16", 0, 2, (6, 12, 136, 184), 115 * 156, 47, 34),
         ("bf16", 0, 0, (13, 5, 27, 47, 57), 27 * 47 * 57, 108, 86), ("fp32", 0, 2, (1, 12, 9, 81, 64), 13 * 117 * 93, 130, 237),
         ("bf16", 0, 2, (12, 31, 18, 62, 20), 18 * 62 * 20, 142, 159), ("fp16", 1, 2, (23, 10, 28, 67, 49), 28 * 67 * 49, 114, 130),
         ("fp32", 1, 0, (10, 2, 14, 26, 17), 14 * 26 * 17, 24, 15),
         # many tiles
         ("fp32", 0, 0, (8, 3, 720, 1280), 720 * 1280, 323, 428), ("fp32", 1, 0, (4, 3, 720, 1280), 720 * 1280, 113, 166),
         ("fp32", 0, 0, (1, 3, 720, 1280), 720 * 1280, 58, 66), ("fp32", 0, 0, (1, 1, 1024, 1024), 512 * 512, 44, 30),
         ("fp32", 0, 0, (4, 3, 1024, 1024), 512 * 512, 114, 118), ("fp32", 0, 0, (1, 3, 704, 1152), 704 * 1152, 54, 50),
         ("fp32", 0, 2, (1, 3, 704, 1152), 704 * 1152, 60, 62), ("fp32", 0, 0, (4, 3, 640, 1120), 640 * 1120, 125, 129),
         ("fp32", 0, 0, (4, 3, 608, 1024), 608 * 1024, 116, 114), ("fp32", 0, 2, (4, 3, 608, 1024), 608 * 1024, 131, 139),
         ("fp32", 0, 2, (4, 3, 600, 800), 600 * 800, 107, 99), ("fp32", 0, 0, (4, 4, 64, 128, 128), 64 * 128 * 128, 300, 461),
         ("fp32", 0, 2, (4, 4, 48, 112, 128), 48 * 112 * 128, 272, 242),
         # border padding, few items and channels
         ("fp32", 0, 1, (2, 3, 248, 464), 248 * 464, 64, 105), ("fp32", 0, 1, (1, 1, 376, 632), 376 * 632, 67, 97),
         ("fp32", 0, 1, (2, 6, 61, 54), 61 * 54, 39, 28), ("bf16", 0, 1, (1, 11, 191, 198), 97 * 100, 39, 27),
         ("fp32", 0, 1, (3, 1, 520, 609), 605 * 708, 674, 380), ("fp32", 0, 1, (5, 2, 405, 480), 405 * 480, 260, 207),
         ("fp32", 1, 1, (1, 2, 368, 624), 368 * 624, 47, 39), ("fp32", 1, 1, (2, 1, 408, 600), 792 * 1164, 540, 153),
         # points at random, and rotated
         ("fp32", 0, 1, (3, 4, 265, 296), 265 * 296, 99, 75), ("fp16", 0, 1, (5, 3, 232, 296), 232 * 296, 110, 78),
         ("fp16", 0, 1, (1, 6, 180, 170), 180 * 170, 38, 33), ("fp32", 0, 1, (1, 3, 384, 552), 461 * 663, 75, 105)]


@pytest.mark.parametrize("dtype,interp,pad,shape,points,lists,tiles", TILES)
def test_sorting_takes_the_faster_of_lists_and_tiles(dtype, interp, pad, shape, points, lists, tiles):
    assert (P.gradient_tiles(dtype, interp, pad, shape, points) is not None) == (tiles < lists)


# (type, padding, items, channels, limit that is the faster, microseconds with it and with the other): volumes, affine grids under
# border padding, of 48 and 96, of 72 and 96; points at random under reflection
CROWDED = [("fp32", 1, 3, 4, 48, 62, 174), ("fp32", 1, 1, 10, 48, 78, 138), ("bf16", 1, 8, 1, 48, 92, 167), ("fp32", 1, 24, 6, 72, 102, 151),
           ("bf16", 1, 13, 5, 72, 117, 151), ("fp16", 2, 3, 6, 96, 104, 163), ("fp16", 2, 2, 16, 96, 88, 132)]


@pytest.mark.parametrize("dtype,pad,n,c,limit,faster,slower", CROWDED)
def test_crowded_tiles_of_volumes_have_the_faster_limit(dtype, pad, n, c, limit, faster, slower):
    assert P.crowded_tiles(dtype, 0, pad, n, c, 3)[1] == limit and faster < slower


def test_gradient_tiles_fit_lds_and_the_launch():
    """2048 tiles of 32 x 16 (16 x 8 x 4) and 2047 blocks of 1024 points an item; a block more for chunks that start at a shift"""
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 16 * 2048, 32), 2000)[2] == 2048
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 16 * 2048 + 1, 32), 2000) is None
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 4 * 32, 8 * 8, 16 * 8), 2000)[2] == 2048
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 4 * 32 + 1, 8 * 8, 16 * 8), 2000) is None
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 832, 1024), 2047 * 1024)[3] == 2047
    assert P.gradient_tiles("fp32", 0, 0, (1, 1, 832, 1024), 2047 * 1024 + 1) is None
    assert P.gradient_tiles("fp32", 0, 0, (128, 1, 9, 20, 21), 3 * 1024, 2)[3] == 4
    assert P.gradient_tiles("fp32", 0, 0, (128, 1, 9, 20, 21), 3 * 1024, 1)[3] == 3
    # bicubic samples have no tiles
    assert P.gradient_tiles("fp32", 2, 0, (1, 1, 64, 64), 2000) is None
    rng = random.Random(10)
    taken = 0
    for _ in range(4000):
        n, c, h, w = (int(2 ** rng.uniform(0, k)) for k in (16, 10, 12, 12))
        shape = (n, c, h, w) if rng.random() < 0.5 else (n, c, int(2 ** rng.uniform(0, 7)), max(1, h // 16), max(1, w // 16))
        p = P.gradient_tiles(rng.choice(["fp32", "fp16", "bf16"]), rng.choice([0, 1]), rng.choice([0, 1, 2]), shape,
                             int(2 ** rng.uniform(8, 21)), rng.choice([1, 1, 3]))
        if p is not None:
            taken += 1
            assert 1 <= p[0] <= n and (p[0] == 1 or p[0] * p[1] * 4 <= 256 << 20) and p[1] * 4 <= 1 << 30
            assert p[2] <= 2048 and p[3] <= 2047 and 1 <= p[4] <= c and p[0] * p[2] * p[4] <= MOST_BLOCKS // 2
    assert taken > 400


# (type, mode, items, plane, points, microseconds in rows and in tiles): measured, bicubic too
GRID = [("fp32", 0, 8, (479, 637), (479, 637), 40.5, 33.2), ("fp16", 0, 6, (576, 472), (362, 297), 15.8, 11.3),
        ("bf16", 0, 2, (90, 146), (90, 146), 19.4, 24.4), ("fp32", 0, 3, (241, 369), (128, 196), 7.0, 7.2),
        ("fp32", 2, 8, (479, 637), (479, 637), 115, 138), ("fp16", 2, 8, (479, 637), (479, 637), 108, 153),
        ("fp32", 2, 2, (720, 1280), (720, 1280), 106, 120), ("fp32", 2, 1, (256, 256), (512, 512), 19.6, 32.3)]


@pytest.mark.parametrize("dtype,interp,n,plane,out,rows,tiles", GRID)
def test_grid_gradient_in_the_faster_of_rows_and_tiles(dtype, interp, n, plane, out, rows, tiles):
    assert (P.grid_gradient_tiles(dtype, interp, n, plane, out) is not None) == (tiles < rows)


def test_grid_gradient_tiles_fit_the_launch():
    # 256 x 256 points: 256 tiles an item
    assert P.grid_gradient_tiles("fp32", 0, 2, (200, 200), (256, 256))[0] == 512
    assert P.grid_gradient_tiles("fp32", 0, MOST_BLOCKS // 256, (200, 200), (256, 256))[1] <= MOST_BLOCKS
    assert P.grid_gradient_tiles("fp32", 0, MOST_BLOCKS // 256 + 1, (200, 200), (256, 256)) is None
    assert P.grid_gradient_tiles("fp32", 0, 2**31 - 1, (200, 200), (40000, 40000)) is None


# (type, image, output, channels last, microseconds before and by runs of rows): measured
NEAREST = [("fp16", (6, 4, 764, 1263), (1528, 2526), False, 117, 42), ("fp32", (17, 11, 62, 120), (151, 292), False, 20.6, 8.1),
           ("bf16", (15, 174, 74, 83), (296, 332), False, 291, 121), ("bf16", (12, 145, 92, 116), (184, 232), True, 166, 35),
           ("fp16", (4, 1, 1004, 1749), (4016, 6996), True, 208, 42), ("fp16", (1, 6, 61, 91), (122, 182), False, 5.0, 6.6),
           ("bf16", (18, 4, 1010, 936), (1078, 999), False, 61.2, 63.7)]


@pytest.mark.parametrize("dtype,shape,out,last,before,runs", NEAREST)
def test_nearest_rows_where_they_are_faster(dtype, shape, out, last, before, runs):
    assert (P.nearest_rows(dtype, shape, out, last) is not None) == (runs < before)


def test_nearest_rows_fit_lds_and_cover_the_row():
    rng = random.Random(11)
    whole = pieces = 0
    for _ in range(4000):
        n, c, h, w = (int(2 ** rng.uniform(0, k)) for k in (6, 9, 11, 12))
        out = tuple(max(v, int(v * rng.uniform(0.9, 5))) for v in (h, w))
        dtype, last = rng.choice(["fp32", "fp16", "bf16"]), rng.random() < 0.5
        p = P.nearest_rows(dtype, (n, c, h, w), out, last)
        if p is not None:
            row = out[1] * (c if last else 1)
            unit = 4 if dtype == "fp32" else 8
            assert p[0] % 8 == 0 and 0 < p[3] <= 64 << 10 and (p[1] - 1) * p[2] < row <= p[1] * p[2]
            assert p[1] == 1 or p[2] % unit == 0
            whole, pieces = whole + (p[1] == 1), pieces + (p[1] > 1)
    assert whole > 300 and pieces > 100


@pytest.mark.parametrize("shape,out,last", [((1, 1001, 40, 40), (80, 80), True), ((1, 1, 8, 1000000), (16, 2000000), False),
                                            ((1, 513, 64, 64), (128, 128), True)])
def test_nearest_rows_plan_takes_no_time(shape, out, last):
    """The plan is made on every call: where no piece of a row fits LDS (the first two) it took 9 us, half as much again as the
    smallest call; 0.1 us, here without optimisation some times that."""
    assert P.nearest_rows_nanoseconds("fp32", shape, out, last) < 2000
