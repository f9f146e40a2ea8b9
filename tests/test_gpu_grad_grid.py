"""Grid gradient of the 2-D sampler a lane per grid point (gs2d_grad.hip): groups of one to eight channels, points in
tiles and in rows, bit for bit against the oracle."""
import numpy as np
import pytest

import inputs as I

pytestmark = pytest.mark.gpu

# tiles: planes beyond 64 KiB and 512 tiles of 16 x 16 points, partial ones along both edges; rows: fewer tiles, smaller
# planes, tiles of which more than a fifth would be padding, a single column (coordinates up to 40000: below fp16's 65504)
TILED = [((2, 1, 191, 177), (256, 257)), ((4, 2, 181, 191), (190, 185)), ((3, 3, 150, 260), (207, 219)),
         ((2, 7, 182, 185), (259, 250)), ((1, 13, 190, 180), (365, 361))]
ROWS = [((1, 5, 181, 191), (125, 131)), ((2, 6, 90, 91), (257, 263)), ((33, 3, 190, 190), (17, 65)), ((1, 11, 40000, 1), (50, 49))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp,pad", [(0, 0), (0, 1), (0, 2), (2, 0), (2, 2)])
@pytest.mark.parametrize("xs,out", TILED + ROWS)
def test_grid_gradient(oracle, device, aclnn, dtype, interp, pad, xs, out):
    import torch
    rng = np.random.default_rng(4300 + 10 * interp + pad)
    x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
    g = I.cast_np(I.affine_grid(rng, xs[0], *out), dtype)
    go = I.cast_np(rng.standard_normal(xs[:2] + out).astype(np.float32), dtype)
    _, ref = oracle.grid_sampler2d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
    _, got = aclnn.grid_sampler2d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad, False,
                                           (False, True))
    torch.cuda.synchronize()
    assert np.array_equal(np.ascontiguousarray(I.from_torch(got, dtype)).view(np.uint8), np.ascontiguousarray(ref).view(np.uint8))
