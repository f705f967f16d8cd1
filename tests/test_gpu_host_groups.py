"""Host-memory batches that the solve reads in place run in the workgroup size
that is fastest there, below four windows for each CU too."""
import time

import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu


def test_in_place_batches_run_in_full_groups(gpu_ctx):
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    rng = numpy.random.default_rng(1)
    d = rng.poisson(40.0, (400, 400)).astype(numpy.float32)
    g = rng.uniform(1.0, 5.0, d.shape).astype(numpy.float32)
    assert _lib.tile_count(*d.shape) <= 4 * 256

    def best(**kw):
        p, out, times = _lib.default_params(**kw), numpy.empty_like(d), []
        for _ in range(200):
            t = time.perf_counter()
            gpu_ctx.reduce_frames([d], [g], [out], [0.1], 0, p)
            times.append(time.perf_counter() - t)
        return min(times), out

    best()
    (t, out), (t4, out4), (t1, out1) = best(), best(waves_per_group=4), best(waves_per_group=1)
    print("default %.0f us, by fours %.0f, by ones %.0f" % (t * 1e6, t4 * 1e6, t1 * 1e6))
    assert numpy.array_equal(out, out4) and numpy.array_equal(out, out1)
    # measured: 1.0, and 1.5 in the groups of one that a batch on the device takes
    assert t <= 1.2 * t4
