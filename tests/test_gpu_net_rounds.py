"""The conv net's forward kernels over several tiles per wave (the next tile's
inputs are loaded while the present tile is in its last layer): every tile has
the result it has when its wave runs nothing else."""
import numpy
import pytest

from ncs_amd import _lib, masks, warmstart

pytestmark = pytest.mark.gpu


def _forward(c, p, x):
    import torch
    n = x.shape[0]
    y = torch.full((n, 16, 16), numpy.nan, device="cuda")
    acts = torch.empty((3, n, 256, 32), dtype=torch.bfloat16, device="cuda")
    _lib.check(c.lib.ncs_hip_net_forward(c.handle, p.data_ptr(), x.data_ptr(), y.data_ptr(),
                                         acts.data_ptr(), n,
                                         torch.cuda.current_stream().cuda_stream), "forward")
    return y, acts


# eight waves a CU take a tile each at first: one tile, a partial workgroup,
# one round exactly, tiles left over after it, a third round
@pytest.mark.parametrize("n", [1, 5, 2048, 2049, 4101])
def test_forward_of_many_tiles_equals_each_alone(gpu_ctx, n):
    import torch
    print("net forward of", n, "tiles", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    p = torch.from_numpy(warmstart.init_params(n, last_scale=1.0)).cuda()
    x = torch.randn((n, 2, 16, 16), generator=gen, device="cuda")
    y, acts = _forward(gpu_ctx, p, x)
    for k in range(0, n, 512):
        yk, ak = _forward(gpu_ctx, p, x[k:k + 512].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(y[k:k + 512], yk)
        assert torch.equal(acts[:, k:k + 512], ak)


def _predict(c, frames):
    import torch
    nt = sum(_lib.tile_count(f["height"], f["width"], f.get("geometry", 0)) for f in frames)
    u0 = torch.full((nt, 256), numpy.nan, device="cuda")
    c.predict_frames_device(frames, u0.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return u0


def _weights(c):
    warmstart.set_context_weights(warmstart.init_params(4, last_scale=1.0))
    c.set_otf_mask(masks.to_fft_order(masks.otf_mask()).astype(numpy.float32))


def _frame(d, g, rows=slice(None), cols=slice(None), geometry=0):
    dv, gv = d[rows, cols], g[rows, cols]
    return dict(data=dv.data_ptr(), gamma=gv.data_ptr(), out=0, height=dv.shape[0],
                width=dv.shape[1], data_stride=dv.stride(0), gamma_stride=gv.stride(0), alpha=0.1,
                geometry=geometry)


def _scene(h, w, seed):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return (50.0 * torch.rand((h, w), generator=gen, device="cuda"),
            2.0 + 8.0 * torch.rand((h, w), generator=gen, device="cuda"))


def test_blocks_of_a_large_frame_equal_their_strips(gpu_ctx):
    """2,900 zero-padded blocks, the last row and column partial, against each
    strip of 16 rows as a frame of its own."""
    import torch
    _weights(gpu_ctx)
    h, w = 790, 923
    d, g = _scene(h, w, 1)
    geo = _lib.GEOM_BLOCKS
    whole = _predict(gpu_ctx, [_frame(d, g, geometry=geo)])
    strips = torch.cat([_predict(gpu_ctx, [_frame(d, g, slice(k, k + 16), geometry=geo)])
                        for k in range(0, h, 16)])
    assert torch.equal(whole, strips)


def test_frames_of_a_batch_equal_each_alone(gpu_ctx):
    """Reference windows and blocks in one launch of several rounds, a frame of
    the smallest side among them, against a launch a frame."""
    import torch
    _weights(gpu_ctx)
    frames, keep = [], []
    for k, (h, w, geo) in enumerate([(700, 701, 0), (15, 15, 0), (61, 300, _lib.GEOM_BLOCKS),
                                     (400, 33, 0), (7, 19, _lib.GEOM_BLOCKS)]):
        d, g = _scene(h, w, 10 + k)
        keep.append((d, g))
        frames.append(_frame(d, g, geometry=geo))
    batch = _predict(gpu_ctx, frames)
    assert torch.equal(batch, torch.cat([_predict(gpu_ctx, [f]) for f in frames]))


def test_backward_clears_and_packs_for_every_caller(gpu_ctx):
    """The gradient does not depend on where the parameters are: a buffer of
    their own, the gradient's own buffer, or the context's weights; without
    tiles it is zero.  One tile: each sum is of one workgroup, in one order."""
    import torch
    host = warmstart.init_params(6, last_scale=1.0)
    p = torch.from_numpy(host).cuda()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    x = torch.randn((1, 2, 16, 16), generator=gen, device="cuda")
    gy = torch.randn((1, 16, 16), generator=gen, device="cuda")
    _, acts = _forward(gpu_ctx, p, x)

    def backward(params, grad, n):
        _lib.check(gpu_ctx.lib.ncs_hip_net_backward(
            gpu_ctx.handle, params, x.data_ptr(), acts.data_ptr(), gy.data_ptr(),
            grad.data_ptr(), None, n, torch.cuda.current_stream().cuda_stream), "backward")
        torch.cuda.synchronize()
        return grad

    ref = backward(p.data_ptr(), torch.full_like(p, 7.0), 1)
    assert float(ref.norm()) > 0.0
    q = p.clone()
    assert torch.equal(backward(q.data_ptr(), q, 1), ref)
    warmstart.set_context_weights(host)
    assert torch.equal(backward(None, torch.full_like(p, 7.0), 1), ref)
    assert not bool(backward(p.data_ptr(), torch.full_like(p, 7.0), 0).any())
