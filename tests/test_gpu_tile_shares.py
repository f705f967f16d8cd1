"""Every tile is solved exactly once however a launch shares them out: all
static (one tile per wave and fewer, remainders, up to 4.5 tiles per wave) and
two fifths static with the rest taken one by one.  waves_per_cu = 1 makes the
edges small: 256 waves on 256 CUs."""
import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiles(gpu_ctx):
    import torch
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    rng = numpy.random.default_rng(5)
    d = torch.from_numpy(rng.poisson(25.0, (3000, 16, 16)).astype(numpy.float32) + 0.5).cuda()
    g = torch.from_numpy(rng.uniform(1.0, 30.0, (3000, 16, 16)).astype(numpy.float32)).cuda()
    return d, g, _solve(gpu_ctx, d, g, 3000)


def _solve(ctx, d, g, n, **kw):
    import torch
    u = torch.full_like(d[:n], -1.0)
    it = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    st = torch.full((n,), -9, dtype=torch.int32, device="cuda")
    ctx.solve_tiles_device(d.data_ptr(), g.data_ptr(), None, u.data_ptr(), it.data_ptr(),
                           st.data_ptr(), None, n, 0.1, _lib.default_params(history=1, **kw),
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return u, it, st


@pytest.mark.parametrize("wpg", [1, 3, 4])
@pytest.mark.parametrize("n", [1, 7, 255, 256, 257, 511, 513, 1151, 1152, 1153, 1161, 1300, 3000])
def test_every_tile_is_solved_once(gpu_ctx, tiles, n, wpg):
    import torch
    d, g, (u0, it0, st0) = tiles
    assert int((st0 != 0).sum()) == 0
    print("tiles", n, "waves per group", wpg, flush=True)
    u, it, st = _solve(gpu_ctx, d, g, n, waves_per_cu=1, waves_per_group=wpg)
    assert torch.equal(u, u0[:n]) and torch.equal(it, it0[:n]) and torch.equal(st, st0[:n])
    # and with the default schedule
    u, it, st = _solve(gpu_ctx, d, g, n)
    assert torch.equal(u, u0[:n]) and torch.equal(it, it0[:n]) and torch.equal(st, st0[:n])
