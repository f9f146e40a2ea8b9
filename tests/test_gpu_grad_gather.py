"""Input gradients of the samplers through the sorting variant (gs_grad_gather.hip), and of planes through the elections
(gs2d_grad.hip) where these are the faster ones, bit for bit against the oracle."""
import numpy as np
import pytest

import host_plans
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


# What the shapes above leave to other variants: bilinear samples of 8 channels and more (the list variant up to 16384
# points) and nearest samples below 25 chunks of points.
SORTED2D = [(0, (1, 70, 20, 31), (130, 140), "random"), (0, (1, 9, 81, 101), (129, 130), "affine"),
            (0, (1, 70, 20, 31), (130, 140), "far"), (1, (2, 3, 37, 53), (82, 81), "affine"),
            (1, (1, 2, 20, 31), (90, 75), "random"), (1, (1, 5, 19, 23), (90, 80), "far"), (1, (2, 9, 81, 101), (81, 101), "affine")]
# Large batches: several chunks of points; planes of two bands, of one and of a few elements that many points share.
ELECTED2D = [(0, (400, 1, 80, 90), (20, 21), "random"), (0, (300, 2, 12, 12), (30, 40), "affine"),
             (1, (600, 1, 12, 12), (90, 80), "random"), (1, (130, 3, 70, 80), (82, 81), "affine"),
             (2, (200, 1, 70, 80), (30, 31), "random"), (2, (300, 2, 16, 16), (45, 50), "affine")]


@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp,xs,out,kind,sorts", [c + (True,) for c in SORTED2D] + [c + (False,) for c in ELECTED2D])
def test_planes_by_the_variant_that_takes_them(oracle, device, aclnn, dtype, interp, xs, out, kind, sorts):
    import torch
    points = out[0] * out[1]
    lists = interp == 0 and xs[1] >= 8 and points <= 16384 and points * (4 if dtype == "fp32" else 2) <= 32768
    assert not lists and (host_plans.sorting_takes_planes(dtype, interp, xs, points) is not None) == sorts
    rng = np.random.default_rng(4050 + interp)
    x = I.cast_np(rng.standard_normal(xs).astype(np.float32), dtype)
    g = I.cast_np(_grid2d(rng, kind, xs[0], *out), dtype)
    go = I.cast_np(rng.standard_normal(xs[:2] + out).astype(np.float32), dtype)
    tensors = [I.to_torch(v, dtype, device) for v in (go, x, g)]
    hs = [aclnn.tensor_handle(t) for t in tensors + tensors[1:]]
    mask = aclnn.create_bool_array([True, False])
    st, ws, ex = aclnn.get_workspace_size_grid_sampler2d_backward(*hs[:3], interp, 1, False, mask, *hs[3:])
    assert st == 0 and (ws > 0) == sorts  # the elections need no workspace
    aclnn.destroy_executor(ex)
    aclnn.destroy_bool_array(mask)
    for h in hs:
        aclnn.destroy_tensor(h)
    for pad in (0, 1, 2):
        ref, _ = oracle.grid_sampler2d_backward(go, x, g, interp, pad, False, dtype=I.oracle_code(dtype))
        got, _ = aclnn.grid_sampler2d_backward(*tensors, interp, pad, False)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref)), pad


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


# contributions of several cells: around the wavefront's steps of 64, and of the parts of 16 that it adds; channels of one
# group of 16 and of two
@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("interp", [0, 2])
@pytest.mark.parametrize("channels,counts", [(1, (33, 47, 48, 49)), (17, (63, 64, 65, 80)), (5, (81, 128, 129, 200))])
def test_crowded_elements(oracle, device, aclnn, dtype, interp, channels, counts):
    import torch
    rng = np.random.default_rng(4090 + interp)
    xs, out = (2, channels, 32, 48), (59, 61)
    at = rng.uniform(0, 1, (xs[0], out[0] * out[1], 2)) * (np.array(xs[:1:-1]) - 1)
    for n in range(xs[0]):
        free = iter(rng.permutation(out[0] * out[1]))
        for e in range(12):
            around = np.array([4 * e + 2, 9 * (e % 3) + 4])
            for _ in range(counts[(e + n) % len(counts)]):
                at[n, next(free)] = around + rng.uniform(-0.9, 0.9, 2)
    g = ((2 * at + 1) / np.array(xs[:1:-1]) - 1).astype(np.float32).reshape((xs[0],) + out + (2,))
    x, g, go = (I.cast_np(v, dtype) for v in (rng.standard_normal(xs).astype(np.float32), g, rng.standard_normal(xs[:2] + out).astype(np.float32)))
    assert host_plans.gradient_tiles(dtype, interp, 1, xs, out[0] * out[1]) is None
    ref, _ = oracle.grid_sampler2d_backward(go, x, g, interp, 1, False, dtype=I.oracle_code(dtype))
    got, _ = aclnn.grid_sampler2d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, 1, False, (True, False))
    torch.cuda.synchronize()
    assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref))


# the same of the eight runs of a voxel: up to 128 are put in order by counting, more by merging; around every other voxel all
# points are in one cell, whose run is sorted apart from 65 on.  Many channels, and more points than the tiles take
@pytest.mark.parametrize("dtype", I.DTYPES)
@pytest.mark.parametrize("xs,out,counts", [((2, 26, 8, 16, 16), (10, 14, 14), (40, 63, 64, 65)), ((1, 2, 6, 12, 12), (9, 14, 14), (100, 126, 127, 128, 129)),
                                           ((1, 3, 6, 12, 12), (20, 20, 20), (130, 190, 260, 700))])
def test_crowded_voxels(oracle, device, aclnn, dtype, xs, out, counts):
    import torch
    rng = np.random.default_rng(4095)
    points, extent = int(np.prod(out)), np.array(xs[:1:-1])
    assert host_plans.gradient_tiles(dtype, 0, 1, xs, points) is None
    at = rng.uniform(0, 1, (xs[0], points, 3)) * (extent - 1)
    for n in range(xs[0]):
        free = iter(rng.permutation(points))
        for e in range(9):
            around = np.array([3 * (e % 3) + 3, 3 * (e // 3) + 3, 3])
            for _ in range(counts[(e + n) % len(counts)]):
                at[n, next(free)] = around + (rng.uniform(0.1, 0.9, 3) if e % 2 else rng.uniform(-0.9, 0.9, 3))
    g = ((2 * at + 1) / extent - 1).astype(np.float32).reshape((xs[0],) + out + (3,))
    x, g, go = (I.cast_np(v, dtype) for v in (rng.standard_normal(xs).astype(np.float32), g, rng.standard_normal(xs[:2] + out).astype(np.float32)))
    ref, _ = oracle.grid_sampler3d_backward(go, x, g, 0, 1, False, dtype=I.oracle_code(dtype))
    with aclnn.option("gs3d_grad_variant", 3):
        got, _ = aclnn.grid_sampler3d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), 0, 1, False, (True, False))
    torch.cuda.synchronize()
    assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref))


def _group(dtype, interp, pad, xs, points, tiles, per_core=1):
    """items that the variant which takes the call runs at a time"""
    by_tiles = host_plans.gradient_tiles(dtype, interp, pad, xs, points, per_core)
    assert (by_tiles is not None) == tiles
    return (by_tiles if tiles else host_plans.gather_groups(dtype, interp, xs, points))[0]


# by lists, which take planes of more tiles than gs_grad_tiles.hip does, and bicubic samples; by tiles
@pytest.mark.parametrize("interp,n,plane,out,tiles", [(0, 13, (1100, 1000), (1090, 1001), False), (2, 9, (480, 641), (500, 641), False),
                                                      (0, 85, (480, 641), (500, 641), True), (1, 97, (700, 700), (701, 699), True)])
def test_planes_in_groups_of_items(device, aclnn, interp, n, plane, out, tiles):
    """a batch whose items are run a group at a time, the last group a shorter one, against its items one by one"""
    import torch
    xs = (n, 1) + plane
    group = _group("fp16", interp, 1, xs, out[0] * out[1], tiles)
    assert group < n and n % group != 0
    g = torch.Generator(device=device).manual_seed(4)
    x = torch.randn(xs, generator=g, device=device).half()
    go = torch.randn((n, 1) + out, generator=g, device=device).half()
    grid = (torch.rand((n,) + out + (2,), generator=g, device=device) * 2.4 - 1.2).half()
    got, _ = aclnn.grid_sampler2d_backward(go, x, grid, interp, 1, False, (True, False))
    for i in range(n):
        one, _ = aclnn.grid_sampler2d_backward(go[i:i + 1], x[i:i + 1], grid[i:i + 1], interp, 1, False, (True, False))
        assert torch.equal(one[0], got[i]), i


@pytest.mark.parametrize("xs,out,tiles", [((299, 1, 9, 20, 21), (39, 32, 31), False), ((129, 1, 25, 70, 75), (25, 69, 77), True)])
def test_volumes_in_groups_of_items(device, aclnn, xs, out, tiles):
    """the chunks of a volume start at a shift that its number in the batch gives, whatever group it is run in"""
    import torch
    n, points = xs[0], out[0] * out[1] * out[2]
    group = _group("fp32", 0, 0, xs, points, tiles, (n + 63) // 64)
    assert group < n and n % group != 0 and points % 256 != 0
    g = torch.Generator(device=device).manual_seed(5)
    x = torch.randn(xs, generator=g, device=device)
    go = torch.randn((n, 1) + out, generator=g, device=device)
    grid = torch.rand((n,) + out + (3,), generator=g, device=device) * 2.2 - 1.1
    grads = []
    for variant in (1, 3):
        with aclnn.option("gs3d_grad_variant", variant):
            grads.append(aclnn.grid_sampler3d_backward(go, x, grid, 0, 0, False, (True, False))[0])
    assert torch.equal(*grads)


@pytest.mark.parametrize("n,plane,tiles", [(13, (1100, 1000), False), (85, (480, 641), True)])
def test_groups_of_items_in_a_graph(device, aclnn, n, plane, tiles):
    """replays of a captured call whose groups share their scratch, with eager work between them"""
    import torch
    xs, out = (n, 1) + plane, plane
    group = _group("fp16", 0, 0, xs, out[0] * out[1], tiles)
    assert group < n and n % group != 0
    g = torch.Generator(device=device).manual_seed(6)
    x, go = (torch.randn(xs, generator=g, device=device).half() for _ in range(2))
    grid = torch.empty((n,) + out + (2,), dtype=torch.float16, device=device)
    dx, dg = torch.empty_like(x), torch.empty_like(grid)
    grids = [(torch.rand(grid.shape, generator=g, device=device) * 2.4 - 1.2).half() for _ in range(3)]
    want = [aclnn.grid_sampler2d_backward(go, x, v) for v in grids]
    grid.copy_(grids[0])
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        aclnn.grid_sampler2d_backward(go, x, grid, input_grad=dx, grid_grad=dg)
        s.synchronize()
        with torch.cuda.graph(graph, stream=s):
            aclnn.grid_sampler2d_backward(go, x, grid, input_grad=dx, grid_grad=dg)
    torch.cuda.synchronize()
    for i in (0, 1, 2, 1):
        grid.copy_(grids[i])
        dx.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dx, want[i][0]) and torch.equal(dg, want[i][1]), i


# the grid gradient of few points, by workgroups of one wavefront: a wavefront's points of two items, an item's workgroups on one
# XCD, the most points of that launch and one row more, eighths of the workgroups that are not as many on every one
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("interp", [0, 2])
@pytest.mark.parametrize("xs,out", [((3, 5, 9, 11), (7, 13)), ((8, 3, 12, 10), (16, 8)), ((8, 9, 20, 31), (64, 64)), ((8, 9, 20, 31), (65, 64)),
                                    ((3, 11, 20, 31), (37, 43))])
def test_grid_gradient_of_few_points(oracle, device, aclnn, dtype, interp, xs, out):
    import torch
    rng = np.random.default_rng(4099 + interp)
    x, go = (I.cast_np(rng.standard_normal(s).astype(np.float32), dtype) for s in (xs, xs[:2] + out))
    g = I.cast_np(_grid2d(rng, "random", xs[0], *out), dtype)
    _, ref = oracle.grid_sampler2d_backward(go, x, g, interp, 0, False, dtype=I.oracle_code(dtype))
    _, got = aclnn.grid_sampler2d_backward(*(I.to_torch(v, dtype, device) for v in (go, x, g)), interp, 0, False, (False, True))
    torch.cuda.synchronize()
    assert np.array_equal(_bits(I.from_torch(got, dtype)), _bits(ref))
