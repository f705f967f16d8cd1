"""Pipelines of one context whose replays take turns on the host link: every
image is bit for bit that of a pipeline alone, however the replays interleave
(waited for one by one, queued deep, on a caller's stream, beside a pipeline
that does other work, from two threads, with one destroyed in between)."""
import threading

import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu

SHAPE = (1480, 1450)  # 8.6 MB an image: just above the size that takes turns
FRAMES = 6


def _pinned(dtype, fill=None):
    import torch
    a = torch.empty(SHAPE, dtype=dtype, pin_memory=True).numpy()
    a[:] = numpy.nan if fill is None else fill
    return a


def _line(ctx, gamma, history=5):
    pl = _lib.Pipeline(ctx, [SHAPE], [0.1], params=_lib.default_params(history=history))
    pl.set_gamma(0, gamma)
    return pl


@pytest.mark.parametrize("mode", ["waited", "deep", "stream", "other", "threads", "destroyed"])
def test_images_are_those_of_a_pipeline_alone(gpu_ctx, mode):
    import torch
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    rng = numpy.random.default_rng(3)
    gamma = (1 + 5 * rng.random(SHAPE)).astype(numpy.float32)
    base = rng.poisson(60, SHAPE).astype(numpy.float32) + 0.5
    ins = [_pinned(torch.float32, numpy.roll(base, 17 * k, 1)) for k in range(FRAMES)]
    want, outs = [_pinned(torch.float32) for _ in ins], [_pinned(torch.float32) for _ in ins]
    alone = _line(gpu_ctx, gamma)
    for a, b in zip(ins, want):
        alone.wait(alone.launch([a], [b]))
    lines = [_line(gpu_ctx, gamma), _line(gpu_ctx, gamma, 2 if mode == "other" else 5)]
    if mode == "other":
        want[1::2] = [_pinned(torch.float32) for _ in want[1::2]]
        for a, b in zip(ins[1::2], want[1::2]):
            lines[1].wait(lines[1].launch([a], [b]))
    if mode == "threads":
        def drive(k):
            for a, b in zip(ins[k::2], outs[k::2]):
                lines[k].wait(lines[k].launch([a], [b]))
        th = [threading.Thread(target=drive, args=(k,)) for k in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    else:
        side = torch.cuda.Stream()
        last = None
        for k, (a, b) in enumerate(zip(ins, outs)):
            pl = lines[k % 2]
            own = mode != "stream" or k % 3 != 1
            seq = pl.launch([a], [b], stream_ptr=None if own else side.cuda_stream)
            if mode == "destroyed" and k == 2:
                lines[0] = _line(gpu_ctx, gamma)
                del pl
                last = None
                continue
            if last is not None and mode != "deep":
                last[0].wait(last[1])
            last = (pl, seq)
        for pl in lines:
            pl.wait()
    torch.cuda.synchronize()
    for a, b in zip(outs, want):
        assert numpy.array_equal(a, b)
