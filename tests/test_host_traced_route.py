"""``torch.jit.trace`` of an operator records one call of its autograd function, which a trace replays on new inputs,
also where nothing needs a gradient."""

import pytest
import torch

from primus_amd.pytorch import ops


class _Opaque(torch.autograd.Function):
    """Its output is written behind torch's back, as by a kernel launch."""

    @staticmethod
    def forward(ctx, x, need_grad=True):
        y = torch.empty_like(x)
        y.numpy()[:] = 2 * x.detach().numpy()
        return y

    @staticmethod
    def backward(ctx, dy):
        return dy * 2.0, None


@pytest.mark.filterwarnings("ignore::DeprecationWarning", "ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("grad", [True, False])
def test_a_trace_replays_on_new_inputs(grad):
    x, z = torch.randn(3, 4), torch.randn(3, 4)
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(lambda t: ops._apply(_Opaque, t), (x,), check_trace=False)
        assert torch.equal(traced(z), 2 * z)
