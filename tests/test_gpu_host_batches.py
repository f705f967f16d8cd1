"""Host-memory batches on both sides of the size where they stop being read in
place (4 MB in and out), with rows that cross the 1 MB staging slots, row
strides, shared and separate gammas and outputs that nobody asked for: bit for
bit the device entry point's results, and nothing written beside them."""
import ctypes

import numpy
import pytest

from ncs_amd import _lib, masks, ncs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx):
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    return gpu_ctx


def _host(h, w, stride, rng):
    a = numpy.full((h, stride), numpy.float32(-7.0))
    a[:, :w] = rng.poisson(25.0, (h, w)).astype(numpy.float32) + 0.5
    return a


def _frame(d, g, o, h, w, alpha):
    f = _lib.Frame()
    f.data, f.gamma = d.ctypes.data, g.ctypes.data
    f.out = None if o is None else o.ctypes.data
    f.height, f.width, f.alpha, f.geometry = h, w, alpha, 0
    f.data_stride, f.gamma_stride = d.shape[1], g.shape[1]
    f.out_stride = 0 if o is None else o.shape[1]
    return f


def _device(ctx, frames):
    """The same frames through the device entry point."""
    import torch
    outs, keep, specs = [], [], []
    for d, g, h, w, a in frames:
        td = torch.from_numpy(numpy.ascontiguousarray(d[:, :w])).cuda()
        tg = torch.from_numpy(numpy.ascontiguousarray(g[:, :w])).cuda()
        to = torch.empty_like(td)
        keep += [td, tg]
        outs.append(to)
        specs.append(dict(data=td.data_ptr(), gamma=tg.data_ptr(), out=to.data_ptr(), height=h,
                          width=w, alpha=a))
    n = sum(_lib.tile_count(h, w) for _, _, h, w, _ in frames)
    it = torch.empty(n, dtype=torch.int32, device="cuda")
    st, co = torch.empty_like(it), torch.empty(n, device="cuda")
    ctx.reduce_frames_device(specs, _lib.default_params(), None, it.data_ptr(), st.data_ptr(),
                             co.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in outs], it.cpu().numpy(), st.cpu().numpy(), co.cpu().numpy()


# (height, width, extra stride) of each frame, one gamma for all
CASES = {
    "one window": [(14, 14, 0)],
    "strided": [(33, 47, 5), (14, 100, 1)],
    # 12 bytes a pixel and 12 a window against 4,194,304: 4,170,096 at
    # 588 x 588, above at 592 x 592
    "last read in place": [(588, 588, 0)],
    "first copied": [(592, 592, 0)],
    "copied, strided": [(592, 592, 3), (40, 30, 7)],
    # over four slots each way, rows of 4804 bytes across their borders
    "many slots": [(1001, 1201, 0), (300, 299, 0)],
}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("shared", [True, False])
def test_host_batch_equals_device_batch(ctx, case, shared):
    print(case, "shared gamma" if shared else "own gammas", flush=True)
    rng = numpy.random.default_rng(len(case))
    frames, arr_o = [], []
    arr = (_lib.Frame * len(CASES[case]))()
    gamma0 = None
    for i, (h, w, extra) in enumerate(CASES[case]):
        d = _host(h, w, w + extra, rng)
        if shared and gamma0 is not None and gamma0.shape == d.shape:
            g = gamma0
        else:
            g = gamma0 = numpy.abs(_host(h, w, w + extra, rng)) * numpy.float32(0.3)
        o = numpy.full((h, w + 2 * extra), numpy.float32(-5.0))
        frames.append((d, g, h, w, 0.1 + 0.05 * i))
        arr_o.append(o)
        arr[i] = _frame(d, g, o, h, w, 0.1 + 0.05 * i)
    n = sum(_lib.tile_count(h, w) for h, w, _ in CASES[case])
    it, st = numpy.full(n + 8, -9, numpy.int32), numpy.full(n + 8, -9, numpy.int32)
    co = numpy.full(n + 8, numpy.float32(-9.0))
    p = _lib.default_params()

    def call(*res):
        _lib.check(ctx.lib.ncs_hip_reduce_frames(
            ctx.handle, arr, len(arr), ctypes.byref(p),
            *[None if r is None else r.ctypes.data for r in res]), "reduce_frames")

    ref, rit, rst, rco = _device(ctx, frames)
    for _ in range(2):
        call(it, st, co)
        for o, r, (d, g, h, w, a) in zip(arr_o, ref, frames):
            assert numpy.array_equal(o[:, :w], r)
            assert numpy.all(o[:, w:] == -5.0)
        assert numpy.array_equal(it[:n], rit) and numpy.array_equal(st[:n], rst)
        assert numpy.array_equal(co[:n], rco)
        assert numpy.all(it[n:] == -9) and numpy.all(st[n:] == -9) and numpy.all(co[n:] == -9.0)
    # some results only, and no image of the last frame
    for o in arr_o:
        o[:] = -5.0
    arr[len(arr) - 1].out = None
    st[:] = -9
    call(None, st, None)
    assert numpy.array_equal(st[:n], rst) and numpy.all(st[n:] == -9)
    for o, r, (d, g, h, w, a) in list(zip(arr_o, ref, frames))[:-1]:
        assert numpy.array_equal(o[:, :w], r)
    assert numpy.all(arr_o[-1] == -5.0)


def test_mask_changes_are_seen(ctx):
    """The tables are kept for a mask of the same values only: another mask,
    its change back, and a change in place of the caller's array all count."""
    rng = numpy.random.default_rng(4)
    im = rng.poisson(25.0, (60, 70)).astype(numpy.float32) + 0.5
    g = rng.uniform(1.0, 20.0, im.shape).astype(numpy.float32)
    a, b = masks.otf_mask(), masks.gaussian_highpass_mask()
    ra = ncs.reduceNoise([im], g, a, 0.1)[0]
    rb = ncs.reduceNoise([im], g, b, 0.1)[0]
    assert not numpy.array_equal(ra, rb)
    assert numpy.array_equal(ncs.reduceNoise([im], g, a, 0.1)[0], ra)
    m = a.copy()
    assert numpy.array_equal(ncs.reduceNoise([im], g, m, 0.1)[0], ra)
    m[:] = b
    assert numpy.array_equal(ncs.reduceNoise([im], g, m, 0.1)[0], rb)
    with pytest.raises(_lib.NCSHipError):
        ctx.set_otf_mask(numpy.full((16, 16), numpy.nan, numpy.float32))
    assert numpy.array_equal(ncs.reduceNoise([im], g, b, 0.1)[0], rb)
    ctx.set_otf_mask(masks.to_fft_order(a).astype(numpy.float32))


def test_a_failed_call_leaves_the_context_usable(ctx):
    im = numpy.full((20, 20), numpy.float32(9.0))
    p = _lib.default_params(start=_lib.START_LEARNED)
    with pytest.raises(_lib.NCSHipError):
        ctx.reduce_frames([im], [im], [numpy.empty_like(im)], [0.1], 0, p)
    out = numpy.empty_like(im)
    ctx.reduce_frames([im], [im], [out], [0.0], 0, _lib.default_params())
    assert numpy.array_equal(out, im)
