"""The reported cost is an evaluation at the returned point: bit for bit what
a solve that starts there and stops there reports, however the search came to
it, and within a bound of the 64-bit cost where the start was a million times
too large."""
import numpy
import pytest

import oracle
from ncs_amd import _lib, linstart, masks

pytestmark = pytest.mark.gpu

N = 200


def _solve(ctx, d, g, u0, alpha, **kw):
    import torch
    t = [None if a is None else torch.as_tensor(a, device="cuda") for a in (d, g, u0)]
    u = torch.empty_like(t[0])
    it = torch.empty(len(d), dtype=torch.int32, device="cuda")
    co = torch.empty(len(d), device="cuda")
    ctx.solve_tiles_device(t[0].data_ptr(), t[1].data_ptr(),
                           None if u0 is None else t[2].data_ptr(), u.data_ptr(),
                           it.data_ptr(), None, co.data_ptr(), len(d), alpha,
                           _lib.default_params(**kw),
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return u.cpu().numpy(), it.cpu().numpy(), co.cpu().numpy()


def _tiles(n):
    rng = numpy.random.default_rng(11)
    d = (rng.poisson(20 + 200 * rng.random((n, 1, 1)), (n, 16, 16)) + 0.5).astype(numpy.float32)
    g = (1 + 10 * rng.random((n, 16, 16))).astype(numpy.float32)
    return d, g


def _context(ctx):
    ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    ctx.set_linear_start(linstart.load(), linstart.load_slope(), 0.1)
    return ctx


@pytest.mark.parametrize("history", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("start,far", [(_lib.START_PLAIN, 1.0), (_lib.START_LINEAR, 1.0),
                                       (_lib.START_PLAIN, 1.02)])
def test_cost_is_evaluated_at_the_returned_point(gpu_ctx, history, start, far):
    ctx = _context(gpu_ctx)
    d, g = _tiles(N)
    u0 = None if far == 1.0 else (d * numpy.float32(far)).astype(numpy.float32)
    u, iters, cost = _solve(ctx, d, g, u0, 0.1, history=history, start=start)
    assert iters.min() >= 1
    # the stop rule holds at once for so large an epsilon
    u2, iters2, cost2 = _solve(ctx, d, g, u, 0.1, history=history, epsilon=1e6, fallback=0)
    assert iters2.max() == 0
    numpy.testing.assert_array_equal(u2, u)
    numpy.testing.assert_array_equal(cost2, cost)


@pytest.mark.parametrize("history", [1, 2, 3, 5, 6, 8])
def test_cost_from_a_start_a_million_times_too_large(gpu_ctx, history):
    ctx = _context(gpu_ctx)
    d, g = _tiles(33)
    alpha = 0.1
    u, _, cost = _solve(ctx, d, g, (d * numpy.float32(1e6)).astype(numpy.float32), alpha,
                        history=history, fallback=0)
    mask = masks.to_fft_order(masks.otf_mask())
    q = numpy.square(mask.astype(numpy.float64))
    for i in range(len(d)):
        p = u[i].astype(numpy.float64)
        v = p + g[i]
        exact, _ = oracle.cost_grad(p, d[i], g[i], mask, alpha)
        # likelihood: 256 terms, 16 roundings each (two operations, a
        # logarithm of four, ten sums)
        terms = numpy.abs(v) + numpy.abs((d[i].astype(numpy.float64) + g[i]) * numpy.log(v))
        # NC = sum q c^2 over the orthonormal coefficients c.  Each c is two
        # sums of 16 products with basis vectors of 1-norm at most 4: off by at
        # most delta = 2 * 16 * 2^-24 * 4 * 4 * max |p|, which for a mean of
        # 1e8 is more than most coefficients themselves.
        delta = 2 * 16 * 2.0 ** -24 * 16 * numpy.abs(p).max()
        nc = numpy.sum(q * numpy.square(numpy.abs(numpy.fft.fft2(p)) / 16.0))
        dn = delta * numpy.sqrt(q.sum())
        tol = 2.0 ** -24 * 16 * terms.sum() + alpha * (2 * numpy.sqrt(nc) * dn + dn * dn)
        assert abs(cost[i] - exact) <= tol, (i, cost[i], exact, tol)
