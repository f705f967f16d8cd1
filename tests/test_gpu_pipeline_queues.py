"""Pairs of like pipelines among more streams than the process has hardware
queues: some of the pairs share a queue, and none of them may lose the overlap
of one replay's transfers with the other's for it."""
import time

import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu

SHAPE = (2304, 2304)
LINES = 5  # one more than the four hardware queues


def test_no_pair_of_like_pipelines_runs_one_after_the_other(gpu_ctx):
    import torch
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    rng = numpy.random.default_rng(2)
    gamma = (1 + 5 * rng.random(SHAPE)).astype(numpy.float32)
    lines = []
    for _ in range(LINES):
        pl = _lib.Pipeline(gpu_ctx, [SHAPE], [0.1])
        pl.set_gamma(0, gamma)
        lines.append(pl)
    pin = lambda: torch.empty(SHAPE, dtype=torch.float32, pin_memory=True).numpy()
    ins, outs = [pin(), pin()], [pin(), pin()]
    for a in ins:
        a[:] = rng.poisson(60, SHAPE).astype(numpy.float32) + 0.5

    def alone(pl):
        t = time.perf_counter()
        for _ in range(6):
            pl.wait(pl.launch([ins[0]], [outs[0]]))
        return time.perf_counter() - t

    def pair(p, q):
        t = time.perf_counter()
        last = None
        for k in range(6):
            now = (p, q)[k % 2]
            seq = now.launch([ins[k % 2]], [outs[k % 2]])
            if last is not None:
                last[0].wait(last[1])
            last = (now, seq)
        last[0].wait(last[1])
        return time.perf_counter() - t

    for pl in lines:
        alone(pl)
    one = min(alone(lines[0]) for _ in range(10))
    worst = 0.0
    for i in range(LINES):
        for j in range(i):
            t = min(pair(lines[j], lines[i]) for _ in range(10))
            print("pipelines", j, i, "%.0f us" % (t * 1e6), flush=True)
            worst = max(worst, t)
    print("one alone %.0f us" % (one * 1e6), flush=True)
    # each direction of the link can carry one replay's copy beside the other's
    # of the other direction; one replay after another takes as long as one
    # pipeline alone (measured: 0.67 to 0.78 of that, and 1.0 with the fault)
    assert worst <= 0.9 * one


def test_uploads_of_like_pipelines_take_turns(gpu_ctx):
    """Of two frames the first has the link to itself on the way up, and is
    solved and on its way down while the second comes."""
    import torch
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    rng = numpy.random.default_rng(2)
    lines = [_lib.Pipeline(gpu_ctx, [SHAPE], [0.1]) for _ in range(LINES)]
    for pl in lines:
        pl.set_gamma(0, numpy.full(SHAPE, 3.0, numpy.float32))
    bufs = [torch.empty(SHAPE, dtype=torch.float32, pin_memory=True).numpy() for _ in range(4)]
    for a in bufs[:2]:
        a[:] = rng.poisson(60, SHAPE).astype(numpy.float32) + 0.5

    def best(p, q):
        times = []
        for _ in range(15):
            t = time.perf_counter()
            first = p.launch([bufs[0]], [bufs[2]])
            if p is q:
                p.wait(first)
            last = q.launch([bufs[1]], [bufs[3]])
            p.wait(first)
            q.wait(last)
            times.append(time.perf_counter() - t)
        return min(times)

    one = min(best(pl, pl) for pl in lines)
    two = min(best(lines[i], lines[j]) for i in range(LINES) for j in range(i))
    print("two frames: one pipeline %.0f us, the best pair %.0f" % (one * 1e6, two * 1e6))
    # measured: 0.77 of one pipeline's time, and 0.92 without the turns
    assert two <= 0.85 * one


def test_replays_of_one_pipeline_wait_for_nothing(gpu_ctx):
    """A lone pipeline, however large its images, makes no stream wait."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    pl = _lib.Pipeline(gpu_ctx, [SHAPE], [0.1])
    pl.set_gamma(0, numpy.ones(SHAPE, numpy.float32))
    a, o = (torch.full(SHAPE, 60.0, dtype=torch.float32, pin_memory=True).numpy() for _ in "ab")
    for _ in range(3):
        pl.wait(pl.launch([a], [o]))
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        for _ in range(4):
            pl.wait(pl.launch([a], [o]))
    calls = [e.name for e in prof.events() if e.name.startswith("hip")]
    print({n: calls.count(n) for n in sorted(set(calls))}, flush=True)
    assert calls.count("hipGraphLaunch") == 4  # the profiler saw the replays
    assert calls.count("hipStreamWaitEvent") == 0
    assert calls.count("hipEventRecord") == 4  # each replay's own
