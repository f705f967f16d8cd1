"""The pinned staging memory of a context follows what its calls need."""
import re

import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu


def _mapped():
    with open("/proc/self/status") as f:
        return int(re.search(r"VmSize:\s+(\d+) kB", f.read()).group(1)) * 1024


def _call(ctx, side):
    rng = numpy.random.default_rng(side)
    d = rng.poisson(30.0, (side, side)).astype(numpy.float32) + 0.5
    g = rng.uniform(1.0, 9.0, d.shape).astype(numpy.float32)
    out = numpy.empty_like(d)
    ctx.reduce_frames([d], [g], [out], [0.1], 0, _lib.default_params(history=1))
    return out


def test_contexts_of_single_windows_pin_little(gpu_ctx):
    m = masks.to_fft_order(masks.otf_mask()).astype(numpy.float32)
    gpu_ctx.set_otf_mask(m)
    _call(gpu_ctx, 14)
    ctxs = [_lib.Context(0) for _ in range(16)]
    try:
        for c in ctxs:
            c.set_otf_mask(m)
        before = _mapped()
        for c in ctxs:
            _call(c, 14)
        grown = _mapped() - before
        print("16 contexts: %.1f MB more mapped" % (grown / 2.0 ** 20))
        # 64 KB a context, and as much again for the allocator's own
        assert grown < 16 * (1 << 20)
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("sides", [(14, 100, 500, 1400, 600, 14), (1400, 14), (75, 73, 75)])
def test_the_staging_grows_between_calls(gpu_ctx, sides):
    m = masks.to_fft_order(masks.otf_mask()).astype(numpy.float32)
    gpu_ctx.set_otf_mask(m)
    ctx = _lib.Context(0)
    try:
        ctx.set_otf_mask(m)
        for side in sides:
            assert numpy.array_equal(_call(ctx, side), _call(gpu_ctx, side)), side
    finally:
        ctx.close()
