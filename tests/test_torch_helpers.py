"""The torch helpers of ops_cv_amd.aclnn beside their results: the streams and the memory that a call uses, and the
arguments that it takes and refuses."""
import pytest


def _block(torch, ptr):
    """(stream of the pool, state) of the caching allocator's block at `ptr`."""
    for seg in torch.cuda.memory_snapshot():
        at = seg["address"]
        for b in seg["blocks"]:
            if at <= ptr < at + b["size"]:
                return seg["stream"], b["state"]
            at += b["size"]
    raise AssertionError("no block at %#x" % ptr)


def _pool_bytes(torch, stream):
    return sum(s["total_size"] for s in torch.cuda.memory_snapshot() if s["stream"] == stream.cuda_stream)


GRADS = ("input_grad", "grid_grad")


def _calls(torch, aclnn, device):
    """name -> (call with further keyword arguments, names of its outputs, whether it needs a workspace)"""
    g = torch.Generator(device=device).manual_seed(5)

    def rand(*shape):
        return torch.rand(shape, generator=g, device=device)
    x, grid, go = rand(2, 3, 40, 50), rand(2, 45, 50, 2) * 2 - 1, rand(2, 3, 45, 50)
    v, vgrid, vgo = rand(2, 3, 8, 20, 20), rand(2, 9, 20, 30, 3) * 2 - 1, rand(2, 3, 9, 20, 30)
    return {
        "sample2d": (lambda **k: aclnn.grid_sampler2d(x, grid, **k), ("out",), False),
        "sample2d_strided": (lambda **k: aclnn.grid_sampler2d(x.transpose(2, 3), grid, **k), ("out",), True),
        "sample2d_grad": (lambda **k: aclnn.grid_sampler2d_backward(go, x, grid, **k), GRADS, True),
        "sample3d": (lambda **k: aclnn.grid_sampler3d(v, vgrid, **k), ("out",), False),
        "sample3d_grad": (lambda **k: aclnn.grid_sampler3d_backward(vgo, v, vgrid, **k), GRADS, True),
        "upsample": (lambda **k: aclnn.upsample_bilinear2d(x, (80, 99), **k), ("out",), False),
        "upsample_grad": (lambda **k: aclnn.upsample_bilinear2d_backward(go, (2, 3, 22, 25), **k), ("out",), False),
        "upsample_grad_dtype": (lambda **k: aclnn.upsample_bilinear2d_backward(go, (2, 3, 22, 25), out_dtype=torch.float16,
                                                                               **k), ("out",), False),
        "nearest": (lambda **k: aclnn.resize(x, (1.0, 1.0, 1.5, 1.5), "nearest", **k), ("out",), False),
    }


CALLS = ["sample2d", "sample2d_strided", "sample2d_grad", "sample3d", "sample3d_grad", "upsample", "upsample_grad",
         "upsample_grad_dtype", "nearest"]


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLS)
def test_memory_of_a_call_on_a_stream_of_its_own(device, aclnn, name):
    """What the call allocates comes from the pool of the stream it runs on, so that no work on the current stream uses
    the memory before, beside or after it; the caller's stream is current again afterwards."""
    import torch
    call, outputs, needs_workspace = _calls(torch, aclnn, device)[name]
    want = call()
    want = want if isinstance(want, tuple) else (want,)
    torch.cuda.synchronize()
    here = torch.cuda.current_stream()
    s = torch.cuda.Stream()
    s.wait_stream(here)
    got = call(stream=s)
    got = got if isinstance(got, tuple) else (got,)
    assert torch.cuda.current_stream() == here
    for t in got:
        assert _block(torch, t.data_ptr())[0] == s.cuda_stream
    here.wait_stream(s)
    for a, b in zip(want, got):
        assert torch.equal(a, b)
    torch.cuda.synchronize()
    if needs_workspace:  # nothing but the workspace is allocated where the caller brings the outputs
        mine = {k: torch.empty_like(t) for k, t in zip(outputs, want)}
        del got, t, b  # the last two by the loops above
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        assert _pool_bytes(torch, s) == 0
        call(stream=s, **mine)
        assert _pool_bytes(torch, s) > 0
        torch.cuda.synchronize()
        for k, a in zip(outputs, want):
            assert torch.equal(mine[k], a)
    with torch.cuda.stream(s):  # a stream that is current already
        again = call(stream=s)
    torch.cuda.synchronize()
    for a, b in zip(want, again if isinstance(again, tuple) else (again,)):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_memory_dropped_while_the_call_waits_on_its_stream(device, aclnn):
    """The caller's operands and workspace, and the outputs that the call made, are not handed out again while the stream
    that uses them still has the call's kernels, or those of the reader, to run."""
    import torch
    g = torch.Generator(device=device).manual_seed(6)
    x = torch.rand((2, 3, 40, 50), generator=g, device=device)
    grid = torch.rand((2, 45, 50, 2), generator=g, device=device) * 2 - 1
    go = torch.rand((2, 3, 45, 50), generator=g, device=device)
    workspace = torch.empty(4 << 20, dtype=torch.uint8, device=device)
    want = aclnn.grid_sampler2d_backward(go, x, grid)
    torch.cuda.synchronize()
    s, here = torch.cuda.Stream(), torch.cuda.current_stream()
    with torch.cuda.stream(s):
        torch.cuda._sleep(200_000_000)  # cycles: the call's kernels wait behind this
    got = aclnn.grid_sampler2d_backward(go, x, grid, stream=s, workspace=workspace)
    at = {"workspace": workspace.data_ptr(), "grad_out": go.data_ptr(), "grid": grid.data_ptr()}
    del workspace, go, grid
    assert not s.query(), "the delay was too short to look behind it"
    for what, ptr in at.items():
        assert _block(torch, ptr)[1] == "active_pending_free", what
    here.wait_stream(s)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    torch.cuda._sleep(200_000_000)  # a reader on the current stream
    ptr = got[0].data_ptr()
    del got
    assert _block(torch, ptr)[1] == "active_pending_free"
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLS)
def test_copy_on_write_outputs_leave_their_source_alone(device, aclnn, name):
    """A lazily cloned tensor that is handed in as an output, or as the workspace, is written into memory of its own."""
    import torch
    call, outputs, needs_workspace = _calls(torch, aclnn, device)[name]
    want = call()
    want = want if isinstance(want, tuple) else (want,)
    sources = {k: torch.full_like(t, 7.0) for k, t in zip(outputs, want)}
    mine = {k: torch._lazy_clone(t) for k, t in sources.items()}
    if needs_workspace:
        sources["workspace"] = torch.full((4 << 20,), 7, dtype=torch.uint8, device=device)
        mine["workspace"] = torch._lazy_clone(sources["workspace"])
    got = call(**mine)
    torch.cuda.synchronize()
    for k, a, b in zip(outputs, want, got if isinstance(got, tuple) else (got,)):
        assert b is mine[k] and torch.equal(a, b)
    for k, t in sources.items():
        assert bool((t == 7).all()), k


@pytest.mark.gpu
def test_arguments_taken_and_refused(device, aclnn):
    """Operands beside a given output are the library's to refuse, with a status; an output that the call would allocate
    needs operands and integers that give its sizes."""
    import numpy as np
    import torch

    def rand(*shape):
        return torch.rand(shape, device=device)
    x, grid, y = rand(1, 2, 9, 10), rand(1, 4, 5, 2), rand(1, 2, 4, 5)
    v, vgrid, vy = rand(1, 2, 3, 9, 10), rand(1, 2, 4, 5, 3), rand(1, 2, 2, 4, 5)
    up = rand(1, 2, 18, 20)

    def status(call):
        with pytest.raises(aclnn.AclnnError) as e:
            call()
        return e.value.status
    INV = aclnn.ACLNN_ERR_PARAM_INVALID
    for few in (x[0], x[0, 0, 0]):
        assert status(lambda: aclnn.grid_sampler2d(few, grid, out=y)) == INV
        assert status(lambda: aclnn.grid_sampler2d(x, few[..., :2], out=y)) == INV
        assert status(lambda: aclnn.grid_sampler3d(few, vgrid, out=vy)) == INV
        assert status(lambda: aclnn.grid_sampler3d(v, few[..., :3], out=vy)) == INV
        assert status(lambda: aclnn.grid_sampler3d(few, vgrid, out=vy, channels_last=True)) == INV
        assert status(lambda: aclnn.upsample_bilinear2d(few, (18, 20), out=up)) == INV
        assert status(lambda: aclnn.resize(few, (1.0, 1.0, 2.0, 2.0), "nearest", out=up)) == INV
    row = x[0, 0, 0]
    for call in (lambda: aclnn.grid_sampler2d(row, grid), lambda: aclnn.grid_sampler2d(x, row),
                 lambda: aclnn.grid_sampler3d(row, vgrid), lambda: aclnn.grid_sampler3d(v, row),
                 lambda: aclnn.upsample_bilinear2d(row, (18, 20)),
                 lambda: aclnn.resize(row, (1.0, 1.0, 2.0, 2.0), "nearest"),
                 lambda: aclnn.upsample_bilinear2d_backward(row, (1, 2, 9, 10))):
        with pytest.raises(IndexError):
            call()
    assert status(lambda: aclnn.upsample_bilinear2d(x, (18,), out=up)) == INV
    assert status(lambda: aclnn.upsample_bilinear2d_backward(up, (1, 2, 9), out=x)) == INV
    # numbers of any kind beside a given output
    want = aclnn.upsample_bilinear2d(x, (18, 20))
    for size in ((18.0, 20.0), [np.int64(18), np.float32(20.5)], np.array([18, 20]), torch.tensor([18, 20]), iter((18, 20))):
        assert torch.equal(aclnn.upsample_bilinear2d(x, size, out=up), want)
    want = aclnn.upsample_bilinear2d_backward(up, (1, 2, 9, 10))
    assert torch.equal(aclnn.upsample_bilinear2d_backward(up, (1, 2.0, np.float64(9), 10.5), out=torch.empty_like(x)), want)
    # integers where they size an allocation
    assert aclnn.upsample_bilinear2d(x, (np.int64(18), 20)).shape == (1, 2, 18, 20)
    for call in (lambda: aclnn.upsample_bilinear2d(x, (18.0, 20)),
                 lambda: aclnn.upsample_bilinear2d_backward(up, (1, 2, 9.0, 10))):
        with pytest.raises(TypeError):
            call()
    with pytest.raises(TypeError):
        aclnn.upsample_bilinear2d_backward(up, (1, 2, 9, 10), out_dtype="float16")
    with pytest.raises(ValueError):
        aclnn.resize(x, (1.0, 1.0, float("nan"), 2.0), "nearest")
    with pytest.raises(OverflowError):
        aclnn.resize(x, (1.0, 1.0, 2.0, float("inf")), "nearest")
    assert aclnn.resize(x, ("1", 1, np.float32(2), "2.0"), "nearest").shape == (1, 2, 18, 20)
    assert torch.equal(aclnn.upsample_bilinear2d(x, (18, 20), False, "2.0", 2), aclnn.upsample_bilinear2d(x, (18, 20)))
    torch.cuda.synchronize()
