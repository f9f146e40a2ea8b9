"""Input gradients of the samplers through the sorting variant (gs_grad_gather.hip), bit for bit against the oracle."""
import numpy as np
import pytest

import inputs as I

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint8)


def _grid2d(rng, kind, n, ho, wo):
    if kind == "affine":
        return I.affine_grid(rng, n, ho, wo)
    if kind == "piled":  # every other column of points on one spot: runs of thousands of entries
        g = rng.uniform(-1.1, 1.1, (n, ho, wo, 2)).astype(np.float32)
        g[:, :, ::2] = 0.3
        return g
    span = 6.0 if kind == "far" else 1.3  # far: most points outside, on the edges under border padding
    return rng.uniform(-span, span, (n, ho, wo, 2)).astype(np.float32)


# (input, grid, kind): partial tiles; one point per element (lists of 16) and more (of 32); elements and runs beyond
# either; channel blocks of 1, 2, 4, 8 and two of 64; for bicubic runs of 16 x 6300 entry values, more than one bitmap
SHAPES2D = [((2, 3, 37, 53), (41, 50), "affine"), ((1, 2, 20, 31), (64, 70), "random"), ((1, 5, 19, 23), (60, 61), "far"),
            ((1, 1, 9, 11), (70, 90), "piled"), ((1, 70, 9, 11), (70, 90), "piled"), ((2, 9, 81, 101), (81, 101), "affine")]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("pad", [0, 1, 2])
def test_planes(oracle, device, aclnn, dtype, interp, pad):
    import torch
    rng = np.random.default_rng(4000 + 10 * interp + pad)
    for (xs, out, kind) in SHAPES2D:
        x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
        g = I.cast_np(_grid2d(rng, kind, xs[0], *out), dtype)
        go = I.cast_np(rng.standard_normal(xs[:2] + out).astype(np.float32), dtype)
        ref, _ = oracle.grid_sampler2d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
        got, _ = aclnn.grid_sampler2d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad, False)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref)), (xs, out, kind)


# the last: more items than the reference device has cores, so that the chunks of every other item start at a shift
SHAPES3D = [((2, 3, 7, 9, 11), (8, 9, 12), 1.1), ((1, 9, 5, 6, 7), (10, 20, 21), 1.1), ((1, 2, 4, 5, 6), (9, 20, 20), 4.0),
            ((70, 1, 3, 4, 5), (3, 10, 10), 1.2)]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("pad", [0, 1, 2])
def test_volumes(oracle, device, aclnn, dtype, interp, pad):
    import torch
    rng = np.random.default_rng(4100 + 10 * interp + pad)
    for (xs, out, span) in SHAPES3D:
        x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
        g = I.cast_np(rng.uniform(-span, span, (xs[0],) + out + (3,)).astype(np.float32), dtype)
        go = I.cast_np(rng.standard_normal(xs[:2] + out).astype(np.float32), dtype)
        ref, _ = oracle.grid_sampler3d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
        with aclnn.option("gs3d_grad_variant", 3):
            got, _ = aclnn.grid_sampler3d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad,
                                                   False)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref)), (xs, out, span)
