"""The window arithmetic at its edges: whole windows (one scalar pointer per
row) against clamped ones, row strides on both sides of the 24-bit limit of
the lane offset, wide frames whose window index is divided by many different
counts, and pixels at the guard beside free ones."""
import numpy
import pytest

from ncs_amd import _lib, linstart, masks

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx):
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    gpu_ctx.set_linear_start(linstart.load(), linstart.load_slope(), 0.1)
    return gpu_ctx


def _scene(h, w, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = torch.poisson(20.0 + 60.0 * torch.rand((h, w), generator=g, device="cuda"), generator=g)
    return d + 0.25, 1.0 + 20.0 * torch.rand((h, w), generator=g, device="cuda")


def _run(ctx, d, g, out, h, w, **kw):
    import torch
    ctx.reduce_frames_device([dict(data=d.data_ptr(), gamma=g.data_ptr(), out=out.data_ptr(),
                                   height=h, width=w, alpha=0.1,
                                   data_stride=d.stride(0), gamma_stride=g.stride(0),
                                   out_stride=out.stride(0))],
                             _lib.default_params(**kw),
                             stream_ptr=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()


def _windows_alone(ctx, d, g, **kw):
    """Every window solved as a tile of its own, stitched on the host."""
    import torch
    h, w = d.shape

    def starts(n):
        return [min(-1 + 14 * i, n - 15) for i in range(1 + -(-(n - 14) // 14))]

    ys, xs = starts(h), starts(w)
    rows = (torch.tensor(ys, device="cuda")[:, None] + torch.arange(16, device="cuda")).clamp(0, h - 1)
    cols = (torch.tensor(xs, device="cuda")[:, None] + torch.arange(16, device="cuda")).clamp(0, w - 1)
    pick = lambda a: a[rows[:, None, :, None], cols[None, :, None, :]].reshape(-1, 16, 16).contiguous()
    dt, gt = pick(d), pick(g)
    u = torch.empty_like(dt)
    ctx.solve_tiles_device(dt.data_ptr(), gt.data_ptr(), None, u.data_ptr(), None, None, None,
                           len(dt), 0.1, _lib.default_params(**kw),
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    u = u.view(len(ys), len(xs), 16, 16).cpu()
    out = torch.zeros((h, w))
    for i, y in enumerate(ys):
        for j, x in enumerate(xs):
            out[y + 1:y + 15, x + 1:x + 15] = u[i, j, 1:15, 1:15]
    return out


@pytest.mark.parametrize("shape", [(14, 14), (15, 16), (16, 15), (28, 29), (30, 42), (43, 58),
                                   (57, 100), (14, 14 * 97 + 5)])
@pytest.mark.parametrize("history", [1, 5])
def test_windows_equal_tiles_solved_alone(ctx, shape, history):
    import torch
    print("frame", shape, "history", history, flush=True)
    d, g = _scene(*shape, seed=sum(shape))
    d[::5, ::7] = 1e-6   # clamped camera pixels with little gamma: at the guard
    g[::5, ::7] = 0.004
    out = torch.full_like(d, -1.0)
    _run(ctx, d, g, out, *shape, history=history)
    ref = _windows_alone(ctx, d, g, history=history)
    # the tile entry point runs the build for padded blocks, whose masked
    # likelihood may round differently: a few last bits of each iteration
    err = float(((out.cpu() - ref).abs() / ref.abs().clamp(min=1.0)).max())
    print("max rel", err, flush=True)
    assert err <= 1e-4


@pytest.mark.parametrize("stride", [(1 << 24) - 1, 1 << 24])
def test_row_strides_around_24_bits(ctx, stride):
    import torch
    h, w = 33, 47
    d, g = _scene(h, w, 7)
    ref = torch.empty_like(d)
    _run(ctx, d, g, ref, h, w, start=_lib.START_LINEAR, history=1)
    big = [torch.empty_strided((h, w), (stride, 1), device="cuda") for _ in range(3)]
    big[0].copy_(d)
    big[1].copy_(g)
    big[2].fill_(-1.0)
    _run(ctx, big[0], big[1], big[2], h, w, start=_lib.START_LINEAR, history=1)
    assert torch.equal(big[2], ref)
    # one of the three strides beyond the limit at a time
    for k in range(3):
        bufs = [d, g, torch.full_like(d, -1.0)]
        bufs[k] = big[k]
        bufs[2].fill_(-1.0)
        _run(ctx, bufs[0], bufs[1], bufs[2], h, w, start=_lib.START_LINEAR, history=1)
        assert torch.equal(bufs[2], ref), k


@pytest.mark.parametrize("windows", [1, 2, 3, 5, 7, 64, 65, 1000, 4097, 9999])
def test_window_index_division(ctx, windows):
    """Two rows of windows and `windows` columns: each column's images of the
    same content are the same."""
    import torch
    h, w = 28, 14 * windows
    d = torch.full((h, w), 20.0, device="cuda")
    d += (torch.arange(w, device="cuda") // 14 % 5).float()[None, :]
    d += (torch.arange(h, device="cuda") // 14 * 3).float()[:, None]
    g = torch.full_like(d, 4.0)
    out = torch.full_like(d, -1.0)
    # alpha 0: the corrected image is the data, so every pixel names its window
    ctx.reduce_frames_device([dict(data=d.data_ptr(), gamma=g.data_ptr(), out=out.data_ptr(),
                                   height=h, width=w, alpha=0.0)], _lib.default_params(),
                             stream_ptr=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(out, d)
