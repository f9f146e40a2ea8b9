"""ctypes view of the kernels' launch plans (host_plans.cpp over the headers of ops_cv_amd/csrc), which need no GPU."""
import ctypes
import os
import subprocess
import tempfile

_HERE = os.path.dirname(os.path.abspath(__file__))
_ROOT = os.path.dirname(_HERE)
ELEM = {"fp32": 0, "fp16": 1, "bf16": 2}
_lib = None


def lib():
    global _lib
    if _lib is None:
        with tempfile.TemporaryDirectory() as d:
            so = os.path.join(d, "libhost_plans.so")
            subprocess.check_call(["g++", "-std=c++17", "-O1", "-ftrapv", "-Wall", "-Wextra", "-shared", "-fPIC",
                                   "-I" + os.path.join(_ROOT, "include"),
                                   "-I" + os.path.join(_ROOT, "ops_cv_amd", "csrc"),
                                   os.path.join(_HERE, "host_plans.cpp"), "-o", so])
            _lib = ctypes.CDLL(so)
    return _lib


def _call(name, count, elem, *args):
    out = (ctypes.c_int64 * count)()
    taken = getattr(lib(), name)(ctypes.c_int(ELEM[elem]), *[ctypes.c_int64(a) for a in args], out)
    return tuple(out) if taken else None


def direct_tiles(dtype, n, c, h, w, ho, wo):
    """(tiles, channel runs) of the direct sampler's tiled kernel, None where it is not taken."""
    return _call("direct_tiles", 2, dtype, n, c, h, w, ho, wo)


def resize_grad_planes(dtype, planes, small, large, align=False):
    """(tile rows, workgroups, planes a workgroup walks at most) of the resize gradient's planes kernel, None where it
    is not taken; the gradient of `small` from `large`, both (rows, columns)."""
    return _call("resize_grad_planes", 3, dtype, planes, *small, *large, int(align))


def resize_grad_rows(dtype, planes, small, large, align=False):
    """(outgoing rows of a wavefront, whether a lane moves two units of a row, rows that an element may visit) of the resize gradient's rows kernel, None where it is not taken."""
    return _call("resize_grad_rows", 3, dtype, planes, *small, *large, int(align))


def resize_grad_kernel(dtype, planes, small, large, align=False):
    """"rows", "planes", "lds" or "gather": the kernel that the resize gradient of dense planes on a 16-byte boundary runs."""
    return (None, "rows", "planes", "lds", "gather")[_call("resize_grad_kernel", 1, dtype, planes, *small, *large, int(align))[0]]


def resize_grad_rows_visits():
    """Most rows, and columns, of the incoming gradient that an outgoing element may visit in the rows kernel."""
    out = (ctypes.c_int64 * 1)()
    assert lib().resize_grad_rows_visits(out) == 1
    return out[0]


def sorting_takes_planes(dtype, interp, shape, points):
    """(elections, sorting): estimated nanoseconds of the input gradient of (N, C, H, W) planes sampled at `points` points
    an item, None where the elections run."""
    return _call("sorting_takes_planes", 2, dtype, interp, *shape, points)


def shrink_in_pairs(unit, rows, shrunk, align=False):
    """Whether channels-last rows of `unit`-byte units shrink two together (resize_nhwc_shrink_kernel)."""
    return bool(lib().shrink_in_pairs(ctypes.c_int64(unit), ctypes.c_int64(rows), ctypes.c_int64(shrunk),
                                      ctypes.c_int(int(align))))


def flat_resize(dtype, planes, small, large):
    """(non-temporal stores, consecutive rows per group) of the flat resize from `small` to `large`."""
    return tuple(bool(v) for v in _call("flat_resize", 2, dtype, planes, *small, *large))


def gather_groups(dtype, interp, shape, points):
    """(items run at a time, 32-bit words of an item) of the sorting input gradient of (N, C, [D,] H, W), None where it
    cannot run."""
    shape = shape if len(shape) == 5 else shape[:2] + (0,) + shape[2:]
    return _call("gather_groups", 2, dtype, interp, *shape, points)


def gradient_tiles(dtype, interp, pad, shape, points, per_core=1):
    """(items run at a time, 32-bit words of an item, tiles, blocks of points, channel blocks) of the sorting input gradient
    by tiles, None where the lists of gather_groups take it."""
    shape = shape if len(shape) == 5 else shape[:2] + (0,) + shape[2:]
    return _call("gradient_tiles", 5, dtype, interp, pad, *shape, points, per_core)


def crowded_tiles(dtype, interp, pad, n, c, dim):
    """(points, contributions of an element) beyond which a tile of the sorting input gradient is a crowded one."""
    return _call("crowded_tiles", 2, dtype, interp, pad, n, c, dim)


def grid_gradient_tiles(dtype, interp, n, plane, out):
    """(tiles, workgroups) of the 2-D sampler's grid gradient, None where its points are taken in rows."""
    return _call("grid_gradient_tiles", 2, dtype, interp, n, *plane, *out)


def nearest_rows(dtype, shape, out, channels_last=False):
    """(rows of a run, pieces of a row, elements of a piece, bytes of LDS) of the nearest resize of (N, C, H, W) images by runs
    of rows, None where another kernel takes it."""
    n, c, h, w = shape
    unit = 4 if dtype == "fp32" else 8
    grid = w * (c if channels_last else 1) % unit == 0 and not (channels_last and c % unit == 0)
    return _call("nearest_rows", 4, dtype, n, c, h, w, *out, int(channels_last), int(grid))


def nearest_rows_nanoseconds(dtype, shape, out, channels_last=False):
    """Host time of that plan."""
    plan = lib().nearest_rows_nanoseconds
    plan.restype = ctypes.c_int64
    return plan(ctypes.c_int(ELEM[dtype]), *[ctypes.c_int64(v) for v in (*shape, *out, int(channels_last))])
