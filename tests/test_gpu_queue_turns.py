"""Solves that take turns with a context's tile counters: launches with and
without dynamic tiles, on two streams, host-memory calls, allocation-free ones
and replays of a captured one in between.  Each gives the bits of the first."""
import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu

# (frames, side): all static; some dynamic tiles; dynamic with a device table
SIZES = [(1, 200), (2, 1800), (34, 420)]


def _batch(n, side, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = torch.poisson(30.0 + 50.0 * torch.rand((n, side, side), generator=g, device="cuda"),
                      generator=g) + 0.5
    return d, 1.0 + 8.0 * torch.rand((n, side, side), generator=g, device="cuda"), d.clone()


def _frames(b):
    d, g, o = b
    return [dict(data=d[i].data_ptr(), gamma=g[i].data_ptr(), out=o[i].data_ptr(),
                 height=d.shape[1], width=d.shape[2], alpha=0.1) for i in range(len(d))]


@pytest.mark.parametrize("order", [
    ("e1", "e1", "e1"),
    ("e1", "e0", "e1", "e2", "e0", "e2"),
    ("e1", "s1", "e1", "s2", "s1"),
    ("c1", "e1", "r1", "e1", "r1", "r1", "e2"),
    ("e1", "h1", "e1", "h0", "e2"),
    ("e1", "n1", "e1", "n1", "e2"),
])
def test_every_solve_gives_the_same_bits(gpu_ctx, order):
    import torch
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    p = _lib.default_params(history=1)
    batches = [_batch(n, s, 7 + s) for n, s in SIZES]
    frames = [_frames(b) for b in batches]
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()

    def eager(k, stream):
        gpu_ctx.reduce_frames_device(frames[k], p, stream_ptr=stream.cuda_stream)

    def noalloc(k, stream):
        arr = _lib.frame_array(frames[k])
        _lib.check(gpu_ctx.lib.ncs_hip_reduce_frames_device_noalloc(
            gpu_ctx.handle, arr, len(arr), p, None, None, None, None,
            stream.cuda_stream), "noalloc")

    want = []
    for k, b in enumerate(batches):
        eager(k, main)
        torch.cuda.synchronize()
        want.append(b[2].clone())
    graphs = {}
    for step in order:
        how, k = step[0], int(step[1])
        out = batches[k][2]
        out.fill_(-1.0)
        torch.cuda.synchronize()
        if how == "e":
            for _ in range(3):
                eager(k, main)
        elif how == "s":
            eager(k, main)
            eager(k, side)
            eager(k, main)
        elif how == "c":
            graphs[k] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graphs[k]):
                noalloc(k, torch.cuda.current_stream())
            graphs[k].replay()
        elif how == "r":
            graphs[k].replay()
            graphs[k].replay()
        elif how == "n":
            noalloc(k, main)
        else:
            d, g, _ = batches[k]
            got = numpy.empty(d.shape, numpy.float32)
            gpu_ctx.reduce_frames(list(d.cpu().numpy()), list(g.cpu().numpy()), list(got),
                                  [0.1] * len(d), 0, p)
            out.copy_(torch.as_tensor(got))
        torch.cuda.synchronize()
        assert torch.equal(out, want[k]), step
