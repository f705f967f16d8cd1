"""The conv net's forward kernel without activations to keep is a build of its
own: bit for bit the outputs of the one that keeps them, at the context's weights
and at a caller's."""
import numpy
import pytest

from ncs_amd import _lib, warmstart

pytestmark = pytest.mark.gpu


# one tile, a partial workgroup, one round exactly, tiles left over, a third round
@pytest.mark.parametrize("n", [1, 5, 2048, 2049, 4101])
def test_outputs_do_not_depend_on_kept_activations(gpu_ctx, n):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n)
    host = warmstart.init_params(n, last_scale=1.0)
    warmstart.set_context_weights(host)
    p = torch.from_numpy(host).cuda()
    x = torch.randn((n, 2, 16, 16), generator=gen, device="cuda")
    acts = torch.empty((3, n, 256, 32), dtype=torch.bfloat16, device="cuda")

    def forward(params, keep):
        y = torch.full((n, 16, 16), numpy.nan, device="cuda")
        _lib.check(gpu_ctx.lib.ncs_hip_net_forward(
            gpu_ctx.handle, None if params is None else params.data_ptr(), x.data_ptr(),
            y.data_ptr(), keep.data_ptr() if keep is not None else None, n,
            torch.cuda.current_stream().cuda_stream), "forward")
        torch.cuda.synchronize()
        return y

    want = forward(p, acts)
    assert not bool(want.isnan().any())
    for params, keep in ((p, None), (None, None), (None, acts)):
        assert torch.equal(forward(params, keep), want)
