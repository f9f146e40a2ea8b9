"""Nearest resize by runs of rows (resize_nearest_rows_kernel), against the oracle."""
import numpy as np
import pytest

import host_plans
import inputs as I

pytestmark = pytest.mark.gpu

# rows off the 16-byte grid and narrow ones on it; runs of 8, 16, 32 and 64 rows, which cross planes and end within one; a
# piece of a row left over; channels of less than a vector and of odd counts; the same height, the same width; whole factors
# that the reference replicates (integer rule) and others.  The third: rows of a run in single precision and in 16 bits, 0
# where another kernel takes the call
PLANES = [((2, 3, 37, 301), (149, 1203), (8, 8)), ((140, 5, 7, 31), (16, 70), (8, 8)), ((4, 3, 301, 333), (301, 999), (8, 8)),
          ((1, 1, 257, 700), (1030, 701), (0, 8)), ((3, 50, 64, 64), (128, 64), (16, 16)), ((1, 700, 3, 5), (41, 33), (16, 16)),
          ((1, 1, 100, 4097), (200, 8194), (8, 8)), ((1, 2, 3, 8191), (70, 16382), (8, 8)), ((300, 1, 1, 33), (19, 99), (8, 8)),
          ((250, 4, 13, 9), (33, 17), (32, 32)), ((500, 4, 13, 5), (33, 9), (64, 64)), ((5, 8, 300, 41), (1700, 82), (64, 64))]
IMAGES = [((5, 3, 57, 61), (171, 244), (8, 8)), ((2, 5, 129, 131), (300, 263), (8, 8)), ((1, 67, 33, 45), (66, 135), (8, 8)),
          ((2, 145, 20, 37), (41, 111), (8, 8)), ((13, 2, 70, 75), (140, 150), (8, 8)), ((1, 33, 5, 300), (205, 600), (0, 8)),
          ((2, 130, 9, 9), (99, 45), (8, 8)), ((5, 3, 300, 41), (7000, 82), (32, 32)), ((700, 3, 13, 5), (97, 9), (64, 64))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,out,runs,last", [c + (False,) for c in PLANES] + [c + (True,) for c in IMAGES])
def test_rows(oracle, device, aclnn, dtype, offset, shape, out, runs, last):
    import torch
    n, c, h, w = shape
    plan = host_plans.nearest_rows(dtype, shape, out, last)
    assert (plan[0] if plan else 0) == runs[0 if dtype == "fp32" else 1]
    rng = np.random.default_rng(4700)
    x = I.cast_np(rng.standard_normal((n, h, w, c) if last else shape).astype(np.float32), dtype)
    t = I.to_torch(x, dtype, device)
    # operands that start on the 16-byte boundary and an element behind it
    xt = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)[offset:offset + t.numel()].view(t.shape).copy_(t)
    ys = (n,) + out + (c,) if last else (n, c) + out
    count = n * c * out[0] * out[1]
    buf = torch.zeros(count + 32, dtype=t.dtype, device=device)
    y = buf[16 + offset:16 + offset + count].view(ys)
    sh, sw = (out[0] + 0.5) / h, (out[1] + 0.5) / w
    aclnn.resize(xt, (1.0, sh, sw, 1.0) if last else (1.0, 1.0, sh, sw), "nearest", channels_last=last, out=y)
    torch.cuda.synchronize()
    ref = oracle.resize_nearest(x, out, channels_last=last, dtype=I.oracle_code(dtype))
    assert np.array_equal(np.ascontiguousarray(I.from_torch(y, dtype)).view(np.uint8), np.ascontiguousarray(ref).view(np.uint8))
    assert not buf[:16 + offset].any() and not buf[16 + offset + count:].any()  # nothing beside the output
