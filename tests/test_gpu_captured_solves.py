"""Solves of the context's own entry point captured into graphs: after a solve
on another stream, replayed between and beside solves outside of the graph, and
two branches of one capture.  Each gives the bits of the plain call."""
import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu


def _batch(n, side):
    import torch
    g = torch.Generator(device="cuda").manual_seed(side)
    d = torch.poisson(30.0 + 50.0 * torch.rand((n, side, side), generator=g, device="cuda"),
                      generator=g) + 0.5
    gamma = 1.0 + 8.0 * torch.rand((n, side, side), generator=g, device="cuda")
    out = torch.empty_like(d)
    frames = [dict(data=d[i].data_ptr(), gamma=gamma[i].data_ptr(), out=out[i].data_ptr(),
                   height=side, width=side, alpha=0.1) for i in range(n)]
    return frames, out, (d, gamma)


@pytest.fixture()
def ctx(gpu_ctx):  # a context of its own: its first solve may be the captured one
    c = _lib.Context(0)
    c.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    yield c
    import torch
    torch.cuda.synchronize()
    c.close()


def _solve(ctx, frames, stream):
    ctx.reduce_frames_device(frames, _lib.default_params(history=1),
                             stream_ptr=stream.cuda_stream)


def _want(frames, out):
    import torch
    c = _lib.Context(0)
    c.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    _solve(c, frames, torch.cuda.current_stream())
    torch.cuda.synchronize()
    c.close()
    return out.clone()


# all tiles static, and some taken from the counters
@pytest.mark.parametrize("captured", [(1, 200), (2, 1800)])
@pytest.mark.parametrize("solve_first", [True, False])
def test_replays_between_other_solves(ctx, captured, solve_first):
    import torch
    frames, out, _k = _batch(*captured)
    other, oout, _k2 = _batch(2, 1500)
    want, owant = _want(frames, out), _want(other, oout)
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    if solve_first:
        _solve(ctx, other, main)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _solve(ctx, frames, torch.cuda.current_stream())
    for stream in (main, side, main):
        out.fill_(-1.0), oout.fill_(-1.0)
        torch.cuda.synchronize()
        _solve(ctx, other, stream)
        graph.replay()
        _solve(ctx, other, stream)
        _solve(ctx, other, main)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(oout, owant)
        out.fill_(-1.0)
        graph.replay()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_two_branches_of_one_capture(ctx):
    import torch
    sets = [_batch(2, 1800), _batch(2, 1700)]
    wants = [_want(f, o) for f, o, _ in sets]
    branch = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        main = torch.cuda.current_stream()
        branch.wait_stream(main)
        _solve(ctx, sets[0][0], main)
        _solve(ctx, sets[1][0], branch)
        main.wait_stream(branch)
    for _ in range(3):
        for _f, o, _k in sets:
            o.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        for (_f, o, _k), w in zip(sets, wants):
            assert torch.equal(o, w)


def test_a_capture_that_needs_the_contexts_table_stays_refused(ctx):
    import torch
    frames, out, _k = _batch(33, 60)
    want = _want(frames, out)
    _solve(ctx, frames, torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _k[0].add_(0.0)  # a graph with a node in it
        with pytest.raises(_lib.NCSHipError, match="captures up to 32 frames"):
            _solve(ctx, frames, torch.cuda.current_stream())
    graph.replay()
    out.fill_(-1.0)
    _solve(ctx, frames, torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(out, want)
