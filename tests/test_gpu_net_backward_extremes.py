"""Layer 4's weight gradient at the ends of FP32: a dL/dout past BF16's
largest value over activations that are zero, activations that are infinite,
and gradients so small that a BF16 remainder of them is subnormal.  Like FP32
products over the in-tile taps: finite where those are, infinite (and not NaN)
where those are, and as close to float64."""
import numpy
import pytest

from ncs_amd import _lib, warmstart

pytestmark = pytest.mark.gpu


def _reference(gy, a3):
    """sum_p dy[p] a3[p + tap][ci] in float64 on the CPU -> [ci, 3, 3]."""
    dy, a = gy.double().cpu().numpy(), a3.double().cpu().numpy().reshape(-1, 16, 16, 32)
    out = numpy.zeros((32, 3, 3))
    for ky in range(3):
        for kx in range(3):
            y0, y1 = max(0, 1 - ky), min(16, 17 - ky)
            x0, x1 = max(0, 1 - kx), min(16, 17 - kx)
            part = a[:, y0 + ky - 1:y1 + ky - 1, x0 + kx - 1:x1 + kx - 1]
            with numpy.errstate(invalid="ignore"):
                out[:, ky, kx] = (dy[:, y0:y1, x0:x1, None] * part).sum(axis=(0, 1, 2))
    return out


@pytest.mark.parametrize("n", [1, 3, 515])
@pytest.mark.parametrize("kind", ["large", "infinite_activation", "tiny"])
def test_layer4_weight_gradient_at_the_ends_of_fp32(gpu_ctx, n, kind):
    import torch
    print("backward,", kind, n, "tiles", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    p = torch.from_numpy(warmstart.init_params(n, last_scale=1.0)).cuda()
    x = torch.randn((n, 2, 16, 16), generator=gen, device="cuda")
    acts = torch.rand((3, n, 256, 32), generator=gen, device="cuda").to(torch.bfloat16)
    gy = torch.rand((n, 16, 16), generator=gen, device="cuda") + 0.5
    if kind == "large":  # one pixel, the largest float, where layer 3 is off
        gy[n - 1, 8, 8] = 3.4028234e38
        acts[2, n - 1].view(16, 16, 32)[7:10, 7:10] = 0.0
        acts[2, n - 1, :, :4] = 0.0
    elif kind == "infinite_activation":  # channel 5, a corner of the last tile
        acts[2, n - 1, 0, 5] = float("inf")
    else:
        gy = gy * 2.0 ** -122
    grad = torch.full_like(p, 7.0)
    c = gpu_ctx
    _lib.check(c.lib.ncs_hip_net_backward(c.handle, p.data_ptr(), x.data_ptr(), acts.data_ptr(),
                                          gy.data_ptr(), grad.data_ptr(), None, n,
                                          torch.cuda.current_stream().cuda_stream), "backward")
    torch.cuda.synchronize()
    ws, bs, _, _ = warmstart.layer_slices()[3]
    got = grad[ws].double().cpu().numpy().reshape(32, 3, 3)
    ref = _reference(gy, acts[2])
    finite = numpy.isfinite(ref)
    assert finite.sum() == (288 if kind != "infinite_activation" else 288 - 4)
    numpy.testing.assert_array_equal(got[~finite], ref[~finite])
    # FP32 sums of at most 256 n positive terms: below 256 roundings a tile and
    # one a tile after that; the products' own rounding is one more
    tol = 2.0 ** -24 * (256 + n + 1) * numpy.abs(ref[finite])
    assert numpy.all(numpy.abs(got[finite] - ref[finite]) <= tol)
