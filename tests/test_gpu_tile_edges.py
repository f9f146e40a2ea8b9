"""Tiled kernels at the edges of their tiles, bit for bit against the oracle: the direct sampler's tiles
(gs2d_kernels.hip), the row groups of the flat resize (resize_flat_lds_kernel.hpp) and the planes variant of the resize
gradient (resize_grad.hip)."""
import numpy as np
import pytest

import host_plans
import inputs as I

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


# (input, output): planes above 32 KiB that no LDS variant takes (odd widths of 16-bit elements, large fp32 planes), few
# output pixels: the row order.  MANY has the tiles: one of 32 x 16 and its remainders; channel runs of 1, 3, 4 + 1 and 18
# times four; two columns
MANY = [((256, 1, 91, 183), (16, 32)), ((43, 3, 91, 183), (33, 65)), ((65, 5, 91, 183), (17, 63)),
        ((2, 70, 91, 183), (31, 97)), ((64, 1, 8201, 2), (40, 37))]
PICTURES = [((1, 5, 301, 211), (16, 32)), ((2, 3, 301, 211), (33, 65)), ((1, 2, 401, 203), (17, 63)),
            ((1, 1, 70001, 2), (40, 37)), ((1, 9, 301, 211), (31, 97))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("align", [False, True])
def test_direct_tiles(oracle, device, aclnn, dtype, interp, pad, align):
    import torch
    rng = np.random.default_rng(5000 + 10 * interp + 2 * pad + align)
    for xs, out in PICTURES:
        x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
        g32 = rng.uniform(-1.3, 1.3, (xs[0],) + out + (2,)).astype(np.float32)
        if interp != 1:  # what a non-finite coordinate gives: the whole pixel NaN
            g32[0, 0, :3, 0] = [np.inf, -np.inf, np.nan]
            g32[0, -1, -3:, 1] = [np.inf, -np.inf, np.nan]
        g32[0, 1, :2] = [[3e38, 0.1], [0.1, -3e38]] if dtype != "fp16" else [[6e4, 0.1], [0.1, -6e4]]
        g = I.cast_np(g32, dtype)
        ref = oracle.grid_sampler2d(x, g, interp, pad, align, dtype=I.oracle_code(dtype))
        with aclnn.option("gs_variant", 1):
            got = aclnn.grid_sampler2d(I.to_torch(x, dtype, device), I.to_torch(g, dtype, device), interp, pad, align)
        torch.cuda.synchronize()
        a, b = I.as_f32(I.from_torch(got, dtype), dtype), I.as_f32(ref, dtype)
        assert np.array_equal(np.isnan(a), np.isnan(b)), (xs, out)
        assert np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)]), (xs, out)


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp,pad", [(0, 0), (0, 1), (0, 2), (1, 0), (1, 1), (1, 2), (2, 1), (2, 2)])
@pytest.mark.parametrize("align", [False, True])
def test_direct_tiles_of_many_pixels(oracle, device, aclnn, dtype, interp, pad, align):
    import torch
    rng = np.random.default_rng(5050 + 10 * interp + 2 * pad + align)
    for xs, out in MANY:
        assert host_plans.direct_tiles(dtype, *xs, *out) is not None
        x = I.cast_np(rng.standard_normal(xs, np.float32), dtype)
        g32 = rng.uniform(-1.3, 1.3, (xs[0],) + out + (2,)).astype(np.float32)
        if interp != 1:  # what a non-finite coordinate gives: the whole pixel NaN
            g32[0, 0, :3, 0] = [np.inf, -np.inf, np.nan]
            g32[-1, -1, -3:, 1] = [np.inf, -np.inf, np.nan]
        # far outside: beyond what an int32 holds, and for 16-bit coordinates as far as they go
        far = {"fp32": 1e10, "bf16": 1e10, "fp16": 6e4}[dtype]
        g32[0, 1, :2] = [[far, 0.1], [0.1, -far]]
        g = I.cast_np(g32, dtype)
        ref = oracle.grid_sampler2d(x, g, interp, pad, align, dtype=I.oracle_code(dtype))
        with aclnn.option("gs_variant", 1):
            got = aclnn.grid_sampler2d(I.to_torch(x, dtype, device), I.to_torch(g, dtype, device), interp, pad, align)
        torch.cuda.synchronize()
        a, b = I.as_f32(I.from_torch(got, dtype), dtype), I.as_f32(ref, dtype)
        assert np.array_equal(np.isnan(a), np.isnan(b)), (xs, out)
        assert np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)]), (xs, out)


# (gradient's planes, size it is reduced to): growth by four (eight visits), three, two, none and a half; one column and
# one row more than a tile of 64 x 16; rows of one element.  Few planes: tiles of 8 rows, each workgroup one plane, and
# 16-bit rows of odd length in the gather; WALKS has the other forms
GROWTH = [((1, 3, 257, 513), (65, 129)), ((300, 1, 67, 259), (17, 65)), ((1, 2, 51, 195), (17, 65)),
          ((2, 3, 33, 129), (16, 64)), ((1, 4, 17, 66), (17, 65)), ((1, 4, 9, 33), (17, 65)), ((1, 1, 4, 1), (3, 1)),
          ((1, 2, 64, 255), (16, 64)), ((1, 2, 31, 511), (16, 128))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("offset", [0, 1])
def test_resize_gradient_planes(oracle, device, aclnn, dtype, align, offset):
    import torch
    rng = np.random.default_rng(5100 + align)
    for gs, small in GROWTH:
        g = I.cast_np(rng.standard_normal(gs).astype(np.float32), dtype)
        ref = oracle.upsample_bilinear2d_backward(g, small, align, dtype=I.oracle_code(dtype))
        t = I.to_torch(g, dtype, device)
        base = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)  # a view that starts off the 4-byte grid
        view = base[offset:].view(t.shape)
        view.copy_(t)
        got = aclnn.upsample_bilinear2d_backward(view, gs[:2] + small, align)
        torch.cuda.synchronize()
        assert _same(I.from_torch(got, dtype), ref), (gs, small)


# (planes, small, large, rows of a tile): workgroups that walk over several planes, the last ones over fewer; tiles of 16
# rows and of 8, cut off at the right and at the bottom; rows of odd length; growth by 1.4, four, 0.6 and two
WALKS = [(701, (40, 70), (57, 101), 16), (211, (65, 129), (257, 513), 8), (905, (70, 131), (45, 79), 16),
         (901, (33, 65), (65, 129), 16)]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("planes,small,large,rows", WALKS)
def test_resize_gradient_planes_in_turn(oracle, device, aclnn, dtype, align, planes, small, large, rows):
    import torch
    tile_rows, blocks, walk = host_plans.resize_grad_planes(dtype, planes, small, large, align)
    assert tile_rows == rows and walk > 1 and planes % walk != 0
    rng = np.random.default_rng(5150 + align)
    g = I.cast_np(rng.standard_normal((1, planes) + large).astype(np.float32), dtype)
    ref = oracle.upsample_bilinear2d_backward(g, small, align, dtype=I.oracle_code(dtype))
    t = I.to_torch(g, dtype, device)
    for offset in (0, 1):  # a view that starts off the 4-byte grid
        base = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        view = base[offset:].view(t.shape)
        view.copy_(t)
        got = aclnn.upsample_bilinear2d_backward(view, (1, planes) + small, align)
        torch.cuda.synchronize()
        assert _same(I.from_torch(got, dtype), ref), offset


# one to seventeen columns past whole tiles (up to four, eight or sixteen are taken a lane per element), more planes than a
# workgroup of them; growth by four, 1.4, 0.6 and none along x
@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("small,wide", [((9, 65), 254), ((5, 66), 92), ((17, 67), 40), ((3, 68), 68), ((6, 69), 270), ((7, 132), 522),
                                        ((5, 80), 310), ((5, 81), 300), ((6, 136), 270), ((4, 144), 130)])
def test_resize_gradient_columns_past_whole_tiles(oracle, device, aclnn, dtype, align, small, wide):
    import torch
    gs = (3, 43, 2 * small[0] + 1, wide)
    assert host_plans.resize_grad_planes(dtype, 129, small, gs[2:], align) is not None
    g32 = np.random.default_rng(5180 + align).standard_normal(gs).astype(np.float32)
    g32[1, 1, 1, -1], g32[2, 5, 2, -2], g32[0, 0, -1, 0] = np.inf, -np.inf, np.nan
    g = I.cast_np(g32, dtype)
    ref = oracle.upsample_bilinear2d_backward(g, small, align, dtype=I.oracle_code(dtype))
    got = aclnn.upsample_bilinear2d_backward(I.to_torch(g, dtype, device), gs[:2] + small, align)
    torch.cuda.synchronize()
    a, b = I.as_f32(I.from_torch(got, dtype), dtype), I.as_f32(ref, dtype)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


# (input, output): groups of consecutive rows with a short last group, a last band of one row, more groups than rows;
# rows that shrink take the groups in turn
FLAT = [((1, 3, 65, 129), (257, 513)), ((2, 40, 7, 9), (29, 31)), ((1, 1, 3, 5), (4, 1000)), ((3, 2, 11, 40), (12, 41)),
        ((1, 7, 33, 50), (20, 77)), ((1, 600, 5, 6), (9, 8))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
def test_flat_resize_groups(oracle, device, aclnn, dtype, align):
    import torch
    rng = np.random.default_rng(5200 + align)
    for xs, out in FLAT:
        x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
        ref = oracle.upsample_bilinear2d(x, out, align, dtype=I.oracle_code(dtype))
        got = aclnn.upsample_bilinear2d(I.to_torch(x, dtype, device), out, align)
        torch.cuda.synchronize()
        assert _same(I.from_torch(got, dtype), ref), (xs, out)


# channels-last images whose rows shrink: units of 4 to 16 bytes, a last band of one, two and three rows, an output row
# longer than a workgroup; a factor just below the rule and one far above it
SHRINK = [((2, 31, 45, 3), (9, 20)), ((1, 24, 1000, 3), (15, 401)), ((1, 40, 30, 1), (10, 13)), ((1, 21, 18, 5), (14, 9)),
          ((2, 50, 33, 2), (6, 33)), ((1, 97, 40, 12), (11, 9)), ((1, 13, 700, 20), (3, 301))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
def test_shrinking_images(oracle, device, aclnn, dtype, align):
    import torch
    rng = np.random.default_rng(5300 + align)
    for xs, out in SHRINK:
        x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
        ref = oracle.upsample_bilinear2d_nhwc(x, out, align, dtype=I.oracle_code(dtype))
        got = aclnn.upsample_bilinear2d(I.to_torch(x, dtype, device), out, align, channels_last=True)
        torch.cuda.synchronize()
        assert _same(I.from_torch(got, dtype), ref), (xs, out)


# (type, planes, small, large, kernel): what resize_grad_rows.hip leaves.  Planes kernel: fp32 rows whose units of 16 bytes are
# estimated at more than two a lane (planes of 42 to 63 columns that grow by three and four), tiles of 8 rows and of 16,
# walked in turn and not, cut off at the bottom; few elements of 16-bit planes of up to three columns; more than 2^18 rows, with one,
# two and eight columns past whole tiles.  Tiles in LDS: growth by more than five along a row, rows of 16 and of 32 bits
LEFT = [("fp32", 2, (13, 56), (52, 224), "planes"), ("fp32", 17, (33, 63), (66, 190), "planes"), ("fp32", 4309, (7, 61), (15, 244), "planes"),
        ("fp32", 1501, (40, 55), (20, 220), "planes"), ("fp32", 5201, (33, 3), (20, 4), "planes"), ("fp16", 4099, (33, 3), (129, 12), "planes"),
        ("bf16", 1337, (96, 2), (336, 8), "planes"), ("fp16", 621, (50, 1), (200, 2), "planes"), ("bf16", 5201, (33, 3), (20, 4), "planes"),
        ("fp16", 1, (2**18 + 3, 66), (2**19 + 9, 131), "planes"), ("bf16", 1, (2**18 + 3, 65), (2**19 + 9, 129), "planes"),
        ("fp32", 1, (2**18 + 3, 72), (3 * 2**18 + 2, 216), "planes"),
        ("fp16", 301, (40, 100), (40, 700), "lds"), ("fp32", 40, (55, 60), (55, 301), "lds"), ("bf16", 64, (37, 200), (28, 1240), "lds")]


@pytest.mark.parametrize("dtype,planes,small,large,kernel", LEFT)
def test_resize_gradient_left_by_rows(oracle, device, aclnn, dtype, planes, small, large, kernel):
    import torch
    assert host_plans.resize_grad_kernel(dtype, planes, small, large) == kernel
    rng = np.random.default_rng(5190)
    g32 = np.resize(rng.standard_normal(1000003).astype(np.float32), (1, planes) + large)
    g32[0, 0, 0, -1], g32[0, -1, 3, -2 if large[1] > 2 else 0], g32[0, planes // 2, -1, 0] = np.inf, -np.inf, np.nan
    g = I.cast_np(g32, dtype)
    ref = oracle.upsample_bilinear2d_backward(g, small, False, dtype=I.oracle_code(dtype))
    t = I.to_torch(g, dtype, device)
    for offset in (0, 1) if planes > 1 and kernel == "planes" else (0,):  # a view that starts off the 16-byte grid
        base = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        view = base[offset:].view(t.shape)
        view.copy_(t)
        got = aclnn.upsample_bilinear2d_backward(view, (1, planes) + small, False)
        torch.cuda.synchronize()
        got, a, b = I.from_torch(got, dtype), I.as_f32(I.from_torch(got, dtype), dtype), I.as_f32(ref, dtype)
        numbers = ~np.isnan(b)
        assert np.array_equal(np.isnan(a), ~numbers) and _same(got[numbers], ref[numbers]), offset
