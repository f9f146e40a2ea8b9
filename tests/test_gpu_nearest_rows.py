"""Nearest resize by runs of rows (resize_nearest_rows_kernel), against the oracle."""
import numpy as np
import pytest

import host_plans
import inputs as I

pytestmark = pytest.mark.gpu

# rows off the 16-byte grid and narrow ones on it; runs that cross planes and end within one; a piece of a row left over;
# channels of less than a vector and of odd counts; the same height, the same width; whole factors that the reference
# replicates (integer rule) and others
PLANES = [((2, 3, 37, 301), (149, 1203)), ((40, 5, 7, 31), (16, 70)), ((1, 3, 301, 333), (301, 999)), ((1, 1, 257, 700), (1030, 701)),
          ((3, 50, 64, 64), (128, 64)), ((1, 700, 3, 5), (41, 33)), ((1, 1, 100, 4097), (200, 8194)), ((1, 2, 3, 8191), (70, 16382)),
          ((300, 1, 1, 33), (19, 99))]
IMAGES = [((2, 3, 57, 61), (171, 244)), ((1, 5, 129, 131), (300, 263)), ((1, 67, 33, 45), (66, 135)), ((2, 145, 20, 37), (41, 111)),
          ((9, 2, 70, 75), (140, 150)), ((1, 33, 5, 300), (205, 600)), ((2, 130, 9, 9), (99, 45))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,out,last", [c + (False,) for c in PLANES] + [c + (True,) for c in IMAGES])
def test_rows(oracle, device, aclnn, dtype, offset, shape, out, last):
    import torch
    n, c, h, w = shape
    small = n * c * out[0] * out[1] * (4 if dtype == "fp32" else 2) < 1 << 20
    assert small or c * w % 4 == 0 or host_plans.nearest_rows(dtype, shape, out, last) is not None
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
