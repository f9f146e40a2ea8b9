"""Input gradients of the samplers by tiles (gs_grad_tiles.hip), bit for bit against the oracle."""
import numpy as np
import pytest

import host_plans
import inputs as I

pytestmark = pytest.mark.gpu


def _check(aclnn, oracle, device, dtype, interp, pad, xs, out, grid, rng, variant=None):
    import torch
    x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
    g = I.cast_np(grid.astype(np.float32), dtype)
    go = I.cast_np(rng.standard_normal(xs[:2] + out).astype(np.float32), dtype)
    if len(xs) == 4:
        ref, _ = oracle.grid_sampler2d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
        got, _ = aclnn.grid_sampler2d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad, False,
                                               (True, False))
    else:
        ref, _ = oracle.grid_sampler3d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
        with aclnn.option("gs3d_grad_variant", 3):
            got, _ = aclnn.grid_sampler3d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad, False,
                                                   (True, False))
    torch.cuda.synchronize()
    a, b = (np.ascontiguousarray(v).view(np.uint8) for v in (I.from_torch(got, dtype), ref))
    assert np.array_equal(a, b), (xs, out)


def _spots(rng, n, count, dim, spread):
    """points on a few spots and scattered ones between them: cells of hundreds of points and elements of thousands"""
    g = rng.uniform(-1.1, 1.1, (n, count, dim))
    at = rng.uniform(-0.9, 0.9, (n, 5, dim))
    for i in range(n):
        some = rng.random(count) < spread
        g[i, some] = at[i, rng.integers(0, 5, int(some.sum()))]
    return g


# tiles of 32 x 16: one, parts of one, edges on and beside their borders; channels together and in blocks (1 to 4, 8 of a
# 16-bit type, several blocks); about one point an element, and a round of points more than LDS holds; the third number:
# points on five spots, so that lanes merge alone (up to 64), the wavefront together, and runs stay single
PLANES = [((1, 1, 16, 32), (40, 41), 0.0), ((2, 3, 49, 65), (47, 61), 0.0), ((3, 2, 33, 95), (50, 61), 0.0),
          ((4, 4, 64, 96), (66, 90), 0.0), ((9, 5, 17, 33), (60, 33), 0.0), ((6, 9, 48, 31), (50, 33), 0.0),
          ((6, 21, 50, 64), (52, 66), 0.0), ((6, 7, 20, 40), (40, 39), 0.9), ((16, 2, 18, 34), (65, 60), 0.5)]

# nearest samples are sorted from 25 chunks of points on
NEAREST = [((1, 1, 80, 96), (90, 100), 0.0), ((8, 3, 97, 130), (70, 99), 0.0), ((9, 9, 65, 95), (81, 83), 0.0),
           ((9, 5, 90, 70), (80, 81), 0.5)]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("interp,xs,out,spots", [(0,) + c for c in PLANES] + [(1,) + c for c in NEAREST])
def test_planes(oracle, device, aclnn, dtype, pad, interp, xs, out, spots):
    rng = np.random.default_rng(4400 + 10 * interp + pad)
    points = out[0] * out[1]
    if spots > 0.0:
        grid = _spots(rng, xs[0], points, 2, spots).reshape((xs[0],) + out + (2,))
    else:
        grid = I.affine_grid(rng, xs[0], *out)
    lists = interp == 0 and xs[1] >= 8 and points % 8 == 0 and points * (4 if dtype == "fp32" else 2) <= 32768
    if pad == 0 and not lists and spots == 0.0:
        assert host_plans.sorting_takes_planes(dtype, interp, xs, points) is not None
        assert host_plans.gradient_tiles(dtype, interp, pad, xs, points) is not None
    _check(aclnn, oracle, device, dtype, interp, pad, xs, out, grid, rng)


# the most tiles, and the most blocks of points, that are taken: counts of all tiles in more than 64 KiB of LDS, and a tile's
# segments found 512 blocks at a time
@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("dtype,xs,out,plan", [("fp32", (1, 1, 1024, 1024), (700, 700), (2048, 479)),
                                               ("fp16", (1, 1, 832, 1024), (1447, 1448), (1664, 2047))])
def test_large_planes(oracle, device, aclnn, interp, dtype, xs, out, plan):
    rng = np.random.default_rng(4550 + interp)
    points = out[0] * out[1]
    assert host_plans.sorting_takes_planes(dtype, interp, xs, points) is not None
    assert host_plans.gradient_tiles(dtype, interp, 0, xs, points)[2:4] == plan
    _check(aclnn, oracle, device, dtype, interp, 0, xs, out, I.affine_grid(rng, 1, *out), rng)


def _cropped(rng, n, out, part, spots):
    """all points on `part` of every axis, some way off the middle, a little turned and jittered; some of them on one spot"""
    axes = [(2 * np.arange(k) + 1) / k - 1 for k in out]
    g = np.stack(np.meshgrid(*axes, indexing="ij")[::-1], axis=-1)
    g[..., 0] += 0.2 * g[..., 1]
    g = g[None] * part + rng.uniform(-0.4, 0.4, (n,) + (1,) * len(out) + (len(out),)) + rng.normal(0, 0.003, (n,) + out + (len(out),))
    some = rng.random(g.shape[:-1]) < spots
    g[some] = 0.3
    return g


# Tiles of many points, which another kernel takes in parts.  Elements with some contributions and with thousands; parts beyond
# the edge of the plane; channels of one workgroup and of several; all points on few elements; chunks at a shift
CROPPED = [((1, 3, 60, 64), (120, 131), 0.25, 0.0), ((2, 1, 20, 37), (93, 101), 0.4, 0.0), ((2, 11, 64, 64), (90, 90), 0.03, 0.1),
           ((3, 2, 100, 90), (93, 96), 0.02, 0.0)]
CROPPED_VOLUMES = [((1, 3, 13, 31, 33), (20, 28, 29), 0.2, 0.0), ((2, 1, 12, 24, 40), (19, 21, 30), 0.15, 0.0), ((1, 8, 30, 30, 30), (29, 28, 31), 0.1, 0.3),
                   ((70, 1, 25, 17, 33), (18, 24, 23), 0.03, 0.1), ((1, 2, 32, 32, 32), (29, 30, 31), 0.01, 0.0)]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("pad", [0, 2])
@pytest.mark.parametrize("xs,out,part,spots", CROPPED + CROPPED_VOLUMES)
def test_crowded_tiles(oracle, device, aclnn, dtype, interp, pad, xs, out, part, spots):
    rng = np.random.default_rng(4580 + interp)
    if interp == 1:
        out = (2 * out[0],) + out[1:]  # of nearest samples a tile may have more points
    grid = _cropped(rng, xs[0], out, part, spots)
    assert host_plans.gradient_tiles(dtype, interp, pad, xs, int(np.prod(out)), 1 if xs[0] < 64 else 2) is not None
    edges, limit = ((32, 16), (5120, 12288)) if len(out) == 2 else ((16, 8, 4), (1920, 10240))
    tile = ((grid + 1) * np.array(xs[:1:-1]) - 1) / 2 // np.array(edges)
    assert any(np.unique(t.reshape(-1, len(out)), axis=0, return_counts=True)[1].max() > limit[interp] for t in tile)
    _check(aclnn, oracle, device, dtype, interp, pad, xs, out, grid, rng)


@pytest.mark.parametrize("n,plane", [(3, (100, 120)), (420, (240, 321))])  # the last: two groups of items, one list after the other
def test_crowded_tiles_in_a_graph(device, aclnn, n, plane):
    """replays of a captured call on grids with crowded tiles and without, with eager work between them"""
    import torch
    rng = np.random.default_rng(4590)
    xs, points = (n, 1) + plane, plane[0] * plane[1]
    group = host_plans.gradient_tiles("fp16", 0, 0, xs, points)[0]
    assert (group < n) == (n == 420) and host_plans.sorting_takes_planes("fp16", 0, xs, points) is not None
    x, go = (torch.from_numpy(rng.standard_normal(xs).astype(np.float16)).to(device) for _ in range(2))
    base = [_cropped(rng, 3, plane, part, 0.0) for part in (0.2, 1.0, 0.05)]
    grids = [torch.from_numpy(g.astype(np.float16)).to(device).repeat(n // 3, 1, 1, 1).contiguous() for g in base]
    want = [aclnn.grid_sampler2d_backward(go, x, g)[0] for g in grids]
    grid, dx, dg = grids[0].clone(), torch.empty_like(x), torch.empty_like(grids[0])
    one, _ = aclnn.grid_sampler2d_backward(go[n - 1:], x[n - 1:], grids[0][n - 1:])
    assert torch.equal(one[0], want[0][n - 1])
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        aclnn.grid_sampler2d_backward(go, x, grid, input_grad=dx, grid_grad=dg)
        s.synchronize()
        with torch.cuda.graph(graph, stream=s):
            aclnn.grid_sampler2d_backward(go, x, grid, input_grad=dx, grid_grad=dg)
    torch.cuda.synchronize()
    for i in (0, 1, 2, 1, 0):
        grid.copy_(grids[i])
        dx.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dx, want[i]), i


# tiles of 16 x 8 x 4; the last two: more items than the reference device has cores, so that the chunks of every other item,
# and with them its blocks of points, start at a shift
VOLUMES = [((1, 1, 4, 8, 16), (8, 8, 9), 0.0), ((2, 3, 5, 9, 17), (8, 9, 12), 0.0), ((1, 4, 9, 17, 33), (9, 17, 33), 0.0),
           ((2, 9, 8, 16, 16), (10, 15, 16), 0.0), ((2, 2, 12, 24, 48), (12, 24, 48), 0.3), ((1, 6, 13, 15, 31), (13, 15, 31), 0.9),
           ((70, 1, 5, 9, 20), (6, 10, 17), 0.0), ((130, 2, 4, 9, 17), (5, 10, 13), 0.2)]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("xs,out,spots", VOLUMES)
def test_volumes(oracle, device, aclnn, dtype, pad, interp, xs, out, spots):
    rng = np.random.default_rng(4500 + 10 * interp + pad)
    points = out[0] * out[1] * out[2]
    if xs[1] <= 8 or interp == 0:
        assert host_plans.gradient_tiles(dtype, interp, pad, xs, points, 1 if xs[0] < 64 else 2) is not None
    if spots > 0.0:
        grid = _spots(rng, xs[0], points, 3, spots)
    else:
        axes = [(2 * np.arange(k) + 1) / k - 1 for k in out]
        z, y, x = np.meshgrid(*axes, indexing="ij")
        grid = np.stack([x, y, z], axis=-1)[None] * rng.uniform(0.9, 1.1, (xs[0], 1, 1, 1, 3)) + rng.normal(0, 0.02, (xs[0],) + out + (3,))
    _check(aclnn, oracle, device, dtype, interp, pad, xs, out, grid.reshape((xs[0],) + out + (3,)), rng)


# Both gradients, that of the grid by workgroups behind the bins of the same launch: points of planes in 16 x 16 tiles, which end
# beside the grid's edges, and in rows; nearest; of volumes the loads of four channels together and, from 262144 points on, of one
BOTH = [(0, (3, 3, 300, 290), (256, 257)), (0, (3, 7, 261, 190), (199, 209)), (0, (3, 2, 33, 95), (50, 61)), (0, (5, 1, 37, 43), (60, 33)),
        (1, (8, 3, 97, 130), (70, 99)), (0, (2, 3, 5, 9, 17), (8, 9, 12)), (0, (2, 9, 8, 16, 16), (10, 15, 16)),
        (0, (9, 3, 33, 32, 32), (29, 32, 33)), (1, (3, 2, 17, 25, 33), (17, 25, 33))]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("interp,xs,out", BOTH)
def test_both_gradients_in_one_launch(oracle, device, aclnn, dtype, pad, interp, xs, out):
    import torch
    rng = np.random.default_rng(4640 + pad)
    points = int(np.prod(out))
    group, _, tiles = host_plans.gradient_tiles(dtype, interp, pad, xs, points)[:3]
    assert group == xs[0] and tiles * 48 <= 40 << 10  # the bins leave room for the grid's workgroups
    if len(xs) == 4:
        in_tiles = interp == 0 and xs[2] * xs[3] > 32768
        assert (host_plans.grid_gradient_tiles(dtype, interp, xs[0], xs[2:], out) is not None) == in_tiles
        backward, reference = aclnn.grid_sampler2d_backward, oracle.grid_sampler2d_backward
        grid = I.affine_grid(rng, xs[0], *out)
    else:
        backward, reference = aclnn.grid_sampler3d_backward, oracle.grid_sampler3d_backward
        axes = [(2 * np.arange(k) + 1) / k - 1 for k in out]
        z, y, x = np.meshgrid(*axes, indexing="ij")
        grid = np.stack([x, y, z], axis=-1)[None] * rng.uniform(0.9, 1.1, (xs[0], 1, 1, 1, 3)) + rng.normal(0, 0.02, (xs[0],) + out + (3,))
    x, g, go = (I.cast_np(v.astype(np.float32), dtype) for v in (rng.standard_normal(xs), grid, rng.standard_normal(xs[:2] + out)))
    ref = reference(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
    with aclnn.option("gs3d_grad_variant", 3 if len(xs) == 5 else 0):
        got = backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, pad, False)
    torch.cuda.synchronize()
    for a, b in zip(got, ref):
        assert np.array_equal(np.ascontiguousarray(I.from_torch(a, dtype)).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


# elements with contributions of several cells, as many as a lane, a wavefront by counting and a wavefront by merging put in
# order: on two elements of a wavefront, and on more than six
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("elements", [2, 9])
@pytest.mark.parametrize("xs,out,counts", [((8, 3, 32, 64), (46, 80), (26, 63, 64, 65)), ((10, 1, 32, 64), (40, 90), (127, 128, 129)),
                                           ((2, 2, 8, 16, 16), (10, 14, 14), (40, 63, 64, 65))])
def test_crowded_elements(oracle, device, aclnn, dtype, elements, xs, out, counts):
    rng = np.random.default_rng(4620)
    points, dim = int(np.prod(out)), len(out)
    assert host_plans.gradient_tiles(dtype, 0, 1, xs, points) is not None
    at = rng.uniform(0, 1, (xs[0], points, dim)) * (np.array(xs[:1:-1]) - 1)
    for n in range(xs[0]):
        free = iter(rng.permutation(points))
        for e in range(elements if dim == 2 else min(elements, 5)):  # of volumes on two planes, in rows of 16
            for row in range(2):
                around = np.array([3 * e + 2, 9 * row + 4] if dim == 2 else [3 * e + 1, 3 * row + 1, 1])
                for _ in range(counts[(e + row + n) % len(counts)]):
                    at[n, next(free)] = around + rng.uniform(-0.9, 0.9, dim)
    grid = (2 * at + 1) / np.array(xs[:1:-1]) - 1
    _check(aclnn, oracle, device, dtype, 0, 1, xs, out, grid.reshape((xs[0],) + out + (dim,)), rng)


# all elements of a row with more contributions than a wavefront takes one after the other, as border padding makes them: a lane
# each; of one element in it as many again as of a dozen others: by the wavefront
@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("xs,out", [((8, 3, 32, 64), (46, 80)), ((3, 9, 48, 64), (50, 64)), ((6, 2, 8, 16, 16), (10, 14, 14))])
@pytest.mark.parametrize("each,most", [(40, 0), (70, 0), (36, 400)])
@pytest.mark.parametrize("edge", [False, True])
def test_crowded_rows(oracle, device, aclnn, dtype, xs, out, each, most, edge):
    rng = np.random.default_rng(4630)
    points, dim = int(np.prod(out)), len(out)
    assert host_plans.gradient_tiles(dtype, 0, 1, xs, points) is not None
    at = rng.uniform(0, 1, (xs[0], points, dim)) * (np.array(xs[:1:-1]) - 1)
    for n in range(xs[0]):
        free = iter(rng.permutation(points))
        # beyond the edge, where border padding takes them to the row of the edge, or around a row inside
        around = np.array([0, -3, -2] if edge else [0, 3, 2])[:dim]
        for x in range(15):
            for _ in range(each + (most if x == n + 2 else 0)):
                at[n, next(free)] = around + np.append(x + rng.uniform(0.1, 0.9), rng.uniform(-0.9, 0.9, dim - 1))
    grid = (2 * at + 1) / np.array(xs[:1:-1]) - 1
    _check(aclnn, oracle, device, dtype, 0, 1, xs, out, grid.reshape((xs[0],) + out + (dim,)), rng)


# border padding of one and two items around the most points that are taken by tiles there, rotated so that points pile up
@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("xs,out,taken", [((1, 6, 190, 180), (180, 182), True), ((2, 2, 190, 180), (180, 182), True), ((1, 6, 180, 190), (182, 181), False)])
def test_border_padding_of_few_items(oracle, device, aclnn, dtype, xs, out, taken):
    rng = np.random.default_rng(4640)
    assert (host_plans.gradient_tiles(dtype, 0, 1, xs, out[0] * out[1]) is not None) == taken
    y, x = np.meshgrid(np.linspace(-1, 1, out[0]), np.linspace(-1, 1, out[1]), indexing="ij")
    turn = np.array([[0.9, -0.5], [0.6, 1.1]])
    grid = np.broadcast_to(np.stack([x, y], -1) @ turn, (xs[0],) + out + (2,)) + rng.uniform(-0.02, 0.02, (xs[0], 1, 1, 2))
    _check(aclnn, oracle, device, dtype, 0, 1, xs, out, grid, rng)


def test_special_grid_values(oracle, device, aclnn):
    """points that are no numbers, infinite or far outside have no tile; on and beside the edges of tiles and of the plane"""
    rng = np.random.default_rng(4600)
    xs, out = (2, 2, 40, 70), (45, 50)
    px = np.concatenate([np.arange(-2, 72, 0.5), [15.999, 31.9999, 32.0001, 63.9999], [np.nan, np.inf, -np.inf, 1e30, -1e30]])
    gx = (2 * rng.choice(px, (2,) + out) + 1) / 70 - 1
    gy = (2 * rng.choice(px, (2,) + out) + 1) / 40 - 1
    for dtype in I.DTYPES:
        for interp, pad in ((0, 0), (0, 2)):
            _check(aclnn, oracle, device, dtype, interp, pad, xs, out, np.stack([gx, gy], axis=-1), rng)
