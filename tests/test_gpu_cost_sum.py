"""The reported cost, carried through the search as the start's cost plus the
steps' sum, against the 64-bit cost of the returned point: near starts and far
ones (which are evaluated afresh), and searches cut short."""
import numpy
import pytest

import oracle
from ncs_amd import _lib, linstart, masks

pytestmark = pytest.mark.gpu

N = 33


def _solve(ctx, d, g, u0, alpha, **kw):
    import torch
    t = [None if a is None else torch.as_tensor(a, device="cuda") for a in (d, g, u0)]
    u = torch.empty_like(t[0])
    st = torch.empty(N, dtype=torch.int32, device="cuda")
    co = torch.empty(N, device="cuda")
    ctx.solve_tiles_device(t[0].data_ptr(), t[1].data_ptr(),
                           None if u0 is None else t[2].data_ptr(), u.data_ptr(), None,
                           st.data_ptr(), co.data_ptr(), N, alpha, _lib.default_params(**kw),
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return u.cpu().numpy(), st.cpu().numpy(), co.cpu().numpy()


@pytest.mark.parametrize("history", [1, 2, 3, 5, 6, 8])
@pytest.mark.parametrize("start,far,kw", [
    (0, 1.0, {}),
    (0, 1.0, dict(max_iterations=2)),
    (0, 1.0, dict(epsilon=0.0, max_iterations=40)),
    (3, 1.0, {}),
    (0, 1.02, {}),
    (0, 30.0, {}),
    # Evaluated afresh.  The bound leaves out what a mean of 1e8 adds to NC: the
    # FP32 basis changes round its leak into the other coefficients, up to
    # 1.5e-5 of the cost, whichever way the cost is formed.
    pytest.param(0, 1e6, {}, marks=pytest.mark.xfail(strict=False, reason="mean's rounding in NC")),
])
def test_cost_is_that_of_the_returned_point(gpu_ctx, history, start, far, kw):
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    gpu_ctx.set_linear_start(linstart.load(), linstart.load_slope(), 0.1)
    rng = numpy.random.default_rng(5)
    d = (rng.poisson(20 + 200 * rng.random((N, 1, 1)), (N, 16, 16)) + 0.5).astype(numpy.float32)
    g = (1 + 10 * rng.random((N, 16, 16))).astype(numpy.float32)
    u0 = None if far == 1.0 else (d * numpy.float32(far)).astype(numpy.float32)
    alpha = 0.1
    u, _, cost = _solve(gpu_ctx, d, g, u0, alpha, history=history, start=start,
                        fallback=int(far == 1.0), **kw)
    mask = masks.to_fft_order(masks.otf_mask())
    for i in range(N):
        p = u[i].astype(numpy.float64)
        v = p + g[i]
        terms = numpy.abs(v) + numpy.abs((d[i].astype(numpy.float64) + g[i]) * numpy.log(v))
        # 256 terms: two FP32 operations and a logarithm each (4 roundings),
        # summed 4 in a lane and over 64 lanes (9 adds), the steps' and the
        # parts' sums (3): 16 roundings.  The start's terms are at most 1.25
        # times the end's before the cost is evaluated afresh, and the start's
        # and the end's errors add: 48.  NC is a sum of squares at FP32 basis
        # changes (16 deep, twice): 64 roundings of |u|'s part in the mask.
        exact, _ = oracle.cost_grad(p, d[i], g[i], mask, alpha)
        tol = 2.0 ** -24 * (48 * terms.sum() + 64 * alpha * numpy.square(p - p.mean()).sum())
        assert abs(cost[i] - exact) <= tol, (i, cost[i], exact, tol)
