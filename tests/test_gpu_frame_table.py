"""Frame tables at the size where they stop travelling with the launch: 32
frames go in the kernel's arguments, 33 through device memory (and past 24 in
two writes of the allocation-free entry point).  Every frame equals itself
solved alone, for each start and entry point."""
import numpy
import pytest

from ncs_amd import _lib, linstart, masks, sim, warmstart

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx):
    gpu_ctx.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))
    gpu_ctx.set_linear_start(linstart.load(), linstart.load_slope(), 0.1)
    warmstart.set_context_weights(warmstart.load())
    return gpu_ctx


@pytest.fixture(scope="module")
def stack():
    import torch
    f = sim.make_frame(17, (90, 120))
    d = torch.from_numpy(f["data"]).cuda()
    g = torch.from_numpy(f["gamma"]).cuda()
    rng = numpy.random.default_rng(2)
    cuts = []
    for _ in range(33):
        h, w = int(rng.integers(14, 60)), int(rng.integers(14, 60))
        y, x = int(rng.integers(0, 90 - h + 1)), int(rng.integers(0, 120 - w + 1))
        cuts.append((y, x, h, w, float(rng.uniform(0.05, 0.3))))
    return d, g, cuts


def _frames(stack, n, outs):
    d, g, cuts = stack
    return [dict(data=d[y:, x:].data_ptr(), gamma=g[y:, x:].data_ptr(), out=o.data_ptr(),
                 height=h, width=w, data_stride=d.shape[1], gamma_stride=g.shape[1], alpha=a)
            for (y, x, h, w, a), o in zip(cuts[:n], outs)]


def _empty(stack, n):
    import torch
    return [torch.full((h, w), -3.0, device="cuda") for _, _, h, w, _ in stack[2][:n]]


@pytest.mark.parametrize("n", [1, 24, 25, 32, 33])
@pytest.mark.parametrize("start", ["plain", "linear", "learned"])
def test_every_frame_of_the_table_is_solved(ctx, stack, n, start):
    import torch
    print("frames", n, start, flush=True)
    p = _lib.default_params(start={"plain": 0, "linear": 3, "learned": 2}[start], history=2)
    s = torch.cuda.current_stream().cuda_stream
    alone = _empty(stack, n)
    for f in _frames(stack, n, alone):
        ctx.reduce_frames_device([f], p, stream_ptr=s)
    torch.cuda.synchronize()
    outs = _empty(stack, n)
    ctx.reduce_frames_device(_frames(stack, n, outs), p, stream_ptr=s)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(outs, alone))
    if start == "learned":
        return
    outs = _empty(stack, n)
    arr = _lib.frame_array(_frames(stack, n, outs))
    _lib.check(ctx.lib.ncs_hip_reduce_frames_device_noalloc(ctx.handle, arr, n, p, None, None,
                                                            None, None, s), "noalloc")
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(outs, alone))
    d, g, cuts = stack
    dn, gn = d.cpu().numpy(), g.cpu().numpy()
    host = [numpy.zeros((h, w), numpy.float32) for _, _, h, w, _ in cuts[:n]]
    ctx.reduce_frames([dn[y:y + h, x:x + w] for y, x, h, w, _ in cuts[:n]],
                      [gn[y:y + h, x:x + w] for y, x, h, w, _ in cuts[:n]], host,
                      [c[4] for c in cuts[:n]], 0, p)
    assert all(numpy.array_equal(a, b.cpu().numpy()) for a, b in zip(host, alone))
