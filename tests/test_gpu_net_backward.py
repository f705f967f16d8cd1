"""The conv net's backward kernel over the tile counts at which its schedule
changes (one tile, an odd team, one round of every workgroup, tiles left over
after it), against float64 sums of the same BF16-rounded operands."""
import numpy
import pytest

from ncs_amd import _lib, warmstart

pytestmark = pytest.mark.gpu


def _shift_sum(dz, a):
    """sum_p dz[p][co] a[p + tap][ci] -> [co, ci, 3, 3]; dz [n, co, 16, 16]."""
    import torch
    ap = torch.nn.functional.pad(a, (1, 1, 1, 1))
    m = dz.permute(1, 0, 2, 3).reshape(dz.shape[1], -1)
    out = torch.empty(dz.shape[1], a.shape[1], 3, 3, dtype=torch.float64, device=a.device)
    for ky in range(3):
        for kx in range(3):
            w = ap[:, :, ky:ky + 16, kx:kx + 16].permute(1, 0, 2, 3).reshape(a.shape[1], -1)
            out[:, :, ky, kx] = m @ w.t().contiguous()
    return out


def _data_grad(dz, w):
    """Gradient of a 3 x 3 convolution's input; w [co, ci, 3, 3]."""
    import torch
    dp = torch.nn.functional.pad(dz, (1, 1, 1, 1))
    out = torch.zeros(dz.shape[0], w.shape[1], 16, 16, dtype=torch.float64, device=dz.device)
    for ky in range(3):
        for kx in range(3):
            part = dp[:, :, 2 - ky:18 - ky, 2 - kx:18 - kx].permute(1, 0, 2, 3)
            got = w[:, :, ky, kx].t().contiguous() @ part.reshape(dz.shape[1], -1)
            out += got.view(w.shape[1], dz.shape[0], 16, 16).permute(1, 0, 2, 3)
    return out


def _reference(params, x, acts, gy):
    """The kernel's rounding points (weights, inputs, data gradients and, for
    layer 4's data gradient, dL/dout in BF16) with float64 sums."""
    import torch
    r = lambda t: t.to(torch.bfloat16).double()
    a = [r(x)] + [acts[k].double().view(-1, 16, 16, 32).permute(0, 3, 1, 2) for k in range(3)]
    g = gy.double()[:, None]
    out = []
    for li in range(3, -1, -1):
        ws, bs, cin, cout = warmstart.layer_slices()[li]
        out.append((_shift_sum(g, a[li]), g.sum(dim=(0, 2, 3))))
        if li > 0:
            w = r(params[ws]).view(cout, cin, 3, 3)
            g = _data_grad(r(g.float()) if li == 3 else g, w) * (a[li] > 0)
            g = r(g.float())
    return list(reversed(out))


@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 1300])
def test_backward_sums_over_every_tile(gpu_ctx, n):
    import torch
    print("backward of", n, "tiles", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(100 + n)
    p = torch.from_numpy(warmstart.init_params(n, last_scale=1.0)).cuda()
    p = p + 0.02 * torch.randn(p.shape, generator=gen, device="cuda")
    x = torch.randn((n, 2, 16, 16), generator=gen, device="cuda")
    # FP32 gradients whose low bits matter: layer 4's weights take them exactly
    gy = torch.randn((n, 16, 16), generator=gen, device="cuda")
    y = torch.empty_like(gy)
    acts = torch.empty((3, n, 256, 32), dtype=torch.bfloat16, device="cuda")
    grad = torch.full_like(p, 7.0)  # overwritten, not added to
    s = torch.cuda.current_stream().cuda_stream
    c = gpu_ctx
    _lib.check(c.lib.ncs_hip_net_forward(c.handle, p.data_ptr(), x.data_ptr(), y.data_ptr(),
                                         acts.data_ptr(), n, s), "forward")
    _lib.check(c.lib.ncs_hip_net_backward(c.handle, p.data_ptr(), x.data_ptr(), acts.data_ptr(),
                                          gy.data_ptr(), grad.data_ptr(), None, n, s), "backward")
    torch.cuda.synchronize()
    for li, (w, b) in enumerate(_reference(p, x, acts, gy)):
        ws, bs, _, _ = warmstart.layer_slices()[li]
        for name, got, ref in (("w", grad[ws], w.reshape(-1)), ("b", grad[bs], b)):
            err = float((got.double() - ref).norm() / ref.norm())
            print("layer", li + 1, name, "rel err", err, flush=True)
            # FP32 sums of 256 n products: below 1e-5.  A data gradient whose
            # FP32 sum lies within about 2^-22 of a BF16 rounding boundary may
            # round the other way (2^-9 of itself, on 1 in 2^13 or so):
            # 2^-9 / sqrt(2^13) = 2e-5 of the tensor.  Layer 4 has none.
            assert err <= (1e-5 if li == 3 else 2e-4), (n, li, name, err)


def test_backward_of_large_gradients_keeps_their_range(gpu_ctx):
    """dL/dout beyond BF16's largest value rounds to infinity in BF16: the
    split of layer 4's weight gradient then keeps that one term (infinite, as
    FP32 sums of such values are), and never turns a finite gradient into
    NaN."""
    import torch
    n = 2
    p = torch.from_numpy(warmstart.init_params(3, last_scale=1.0)).cuda()
    x = torch.rand((n, 2, 16, 16), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    y = torch.empty((n, 16, 16), device="cuda")
    acts = torch.empty((3, n, 256, 32), dtype=torch.bfloat16, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    c = gpu_ctx
    _lib.check(c.lib.ncs_hip_net_forward(c.handle, p.data_ptr(), x.data_ptr(), y.data_ptr(),
                                         acts.data_ptr(), n, s), "forward")
    for scale in (1e-30, 1e30):
        gy = torch.full((n, 16, 16), scale, device="cuda")
        grad = torch.empty_like(p)
        _lib.check(c.lib.ncs_hip_net_backward(c.handle, p.data_ptr(), x.data_ptr(),
                                              acts.data_ptr(), gy.data_ptr(), grad.data_ptr(),
                                              None, n, s), "backward")
        torch.cuda.synchronize()
        assert bool(torch.isfinite(grad).all())
        w4 = grad[warmstart.layer_slices()[3][0]].double() / scale
        ref = _shift_sum(torch.ones((n, 1, 16, 16), device="cuda", dtype=torch.float64),
                         acts[2].double().view(-1, 16, 16, 32).permute(0, 3, 1, 2)).reshape(-1)
        assert float((w4 - ref).norm() / ref.norm()) <= 1e-5
    assert numpy.isfinite(float(y.sum()))
