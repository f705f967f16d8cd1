"""The default workgroup of four waves at the depths where its LDS is largest
(history 8 with the FP16 split takes just over 64 KB): the bits of one wave per
workgroup."""
import numpy
import pytest

from ncs_amd import _lib, masks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [_lib.PRECISION_FP32, _lib.PRECISION_F16_SPLIT])
@pytest.mark.parametrize("geometry", [_lib.GEOM_REFERENCE, _lib.GEOM_BLOCKS])
@pytest.mark.parametrize("history", [4, 8])
def test_deep_histories_in_default_groups(gpu_ctx, history, geometry, precision):
    import torch
    mask = masks.otf_mask()
    gpu_ctx.set_otf_mask(masks.to_fft_order(mask).astype(numpy.float32))
    shape = (700, 900)  # over four windows or blocks for each of 256 CUs
    assert _lib.tile_count(*shape, geometry) > 4 * 256
    rng = numpy.random.default_rng(history)
    d = torch.from_numpy(rng.poisson(30.0, shape).astype(numpy.float32) + 0.5).cuda()
    g = torch.from_numpy(rng.uniform(1.0, 9.0, shape).astype(numpy.float32)).cuda()

    def solve(**kw):
        out = torch.full_like(d, -1.0)
        frame = dict(data=d.data_ptr(), gamma=g.data_ptr(), out=out.data_ptr(), height=shape[0],
                     width=shape[1], alpha=0.1, geometry=geometry)
        gpu_ctx.reduce_frames_device(
            [frame], _lib.default_params(history=history, precision=precision, **kw),
            stream_ptr=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return out

    one = solve(waves_per_group=1)
    assert torch.equal(solve(), one)
    assert torch.equal(solve(waves_per_group=4), one)
