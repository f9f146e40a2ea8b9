"""Resize gradient of planes with incoming rows in registers (resize_grad_rows.hip), bit for bit against the oracle."""
import numpy as np
import pytest

import host_plans
import inputs as I

pytestmark = pytest.mark.gpu

# ((N, C, rows, columns) of the incoming gradient, size it is reduced to): wavefronts over parts of two planes and over many
# planes, whole and cut; runs of 2, 4, 6, 8 and 10 columns, wider than the plane too; growth by three, whose integer
# coordinates three outgoing rows may visit; nine and ten rows (corners aligned, growth by four); a lane's two units; shrinking;
# two to 64 rows a wavefront
CASES = [((2, 3, 129, 259), (43, 65)), ((5, 7, 28, 27), (14, 9)), ((3, 50, 13, 11), (7, 4)), ((9, 40, 9, 5), (4, 5)),
         ((1, 2, 193, 195), (65, 65)), ((2, 2, 20, 80), (5, 20)), ((1, 3, 64, 64), (16, 16)), ((1, 1, 259, 1021), (65, 256)),
         ((1, 2, 31, 100), (77, 250)), ((1, 1, 5, 6), (40, 37)), ((1, 1, 1, 1), (9, 70)), ((1, 1, 2, 3), (1, 1)),
         ((13, 150, 34, 40), (67, 33)), ((1, 400, 90, 130), (45, 128))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("gs,small", CASES)
def test_rows(oracle, device, aclnn, dtype, align, gs, small):
    import torch
    # rows of a wavefront, two units a lane, more than eight rows; None where another kernel takes it
    plan = host_plans.resize_grad_rows(dtype, gs[0] * gs[1], small, gs[2:], align)
    assert plan is not None or small[1] < 4 or align and 1 in small + gs[2:]
    rng = np.random.default_rng(5300 + align)
    g32 = rng.standard_normal(gs).astype(np.float32)
    # what a lane reads beyond its own columns counts for nothing
    g32[rng.random(gs) < 1e-3] = np.inf
    g32[rng.random(gs) < 1e-3] = np.nan
    g = I.cast_np(g32, dtype)
    ref = oracle.upsample_bilinear2d_backward(g, small, align, dtype=I.oracle_code(dtype))
    t = I.to_torch(g, dtype, device)
    for offset in (0, 1):  # a view that starts off the 16-byte grid
        base = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        view = base[offset:].view(t.shape)
        view.copy_(t)
        got = aclnn.upsample_bilinear2d_backward(view, gs[:2] + small, align)
        torch.cuda.synchronize()
        a, b = I.as_f32(I.from_torch(got, dtype), dtype), I.as_f32(ref, dtype)
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)]), offset


def _check(oracle, device, aclnn, dtype, align, gs, small):
    """raw bits, but for what a NaN holds: whether a sum of zeros keeps its sign too"""
    import torch
    rng = np.random.default_rng(5300 + align)
    g32 = rng.standard_normal(gs).astype(np.float32)
    g32[rng.random(gs) < 1e-3] = np.inf
    g32[rng.random(gs) < 1e-3] = np.nan
    g32[rng.random(gs) < 0.3] = -0.0
    g = I.cast_np(g32, dtype)
    ref = oracle.upsample_bilinear2d_backward(g, small, align, dtype=I.oracle_code(dtype))
    t = I.to_torch(g, dtype, device)
    for offset in (0, 1):  # a view that starts off the 16-byte grid
        base = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        view = base[offset:].view(t.shape)
        view.copy_(t)
        got = I.from_torch(aclnn.upsample_bilinear2d_backward(view, gs[:2] + small, align), dtype)
        torch.cuda.synchronize()
        numbers = ~np.isnan(I.as_f32(ref, dtype))
        assert np.array_equal(~np.isnan(I.as_f32(got, dtype)), numbers), offset
        assert np.array_equal(np.ascontiguousarray(got[numbers]).view(np.uint8), np.ascontiguousarray(ref[numbers]).view(np.uint8)), offset


# of the cases above those that have too few elements for the rows kernel, with more planes; growth by 4.7
MORE = [((5, 170, 28, 27), (14, 9)), ((3, 700, 13, 11), (7, 4)), ((9, 2000, 9, 5), (4, 5)), ((1, 24, 31, 100), (77, 250)),
        ((3, 120, 5, 6), (40, 37)), ((8, 100, 1, 1), (9, 70)), ((2, 3, 129, 259), (43, 65)), ((1, 2, 193, 195), (65, 65)),
        ((13, 150, 34, 40), (67, 33)), ((3, 7, 98, 78), (21, 17))]
# growth by five, eleven rows, columns or both
FIVE = [(False, (2, 5, 75, 325), (15, 65)), (True, (1, 3, 66, 321), (14, 65)), (False, (1, 3, 200, 40), (40, 8)), (True, (40, 1, 161, 43), (33, 43)),
        (True, (3, 100, 17, 326), (33, 66)), (False, (1, 1, 505, 500), (101, 100))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("gs,small", MORE)
def test_rows_of_many_planes(oracle, device, aclnn, dtype, align, gs, small):
    assert host_plans.resize_grad_kernel(dtype, gs[0] * gs[1], small, gs[2:], align) == "rows" or align and 1 in small + gs[2:]
    _check(oracle, device, aclnn, dtype, align, gs, small)


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("align,gs,small", FIVE)
def test_growth_by_five(oracle, device, aclnn, dtype, align, gs, small):
    assert host_plans.resize_grad_kernel(dtype, gs[0] * gs[1], small, gs[2:], align) == "rows"
    assert host_plans.resize_grad_rows(dtype, gs[0] * gs[1], small, gs[2:], align)[2] == 12
    _check(oracle, device, aclnn, dtype, align, gs, small)


def test_a_row_refused_behind_others(oracle, device, aclnn):
    """growth by a little less than four, eight visits but for row 2060 of 2354, which rounding gives nine: the wavefronts of 16
    rows that hold it have stored twelve when they find out, and have taken the weights of eight more"""
    gs, small = (1, 27, 9412, 64), (2354, 257)
    assert host_plans.resize_grad_kernel("fp16", 27, small, gs[2:]) == "rows" and host_plans.resize_grad_rows("fp16", 27, small, gs[2:]) == (16, 0, 8)
    _check(oracle, device, aclnn, "fp16", False, gs, small)
