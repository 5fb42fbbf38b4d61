"""The route that leaves the autograd function out where nothing needs a gradient: taken for plain tensors only."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from primus_amd.pytorch import ops


class _Twice(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, need_grad=True):
        with torch.no_grad():
            y = x.detach() * 2.0
        ctx.save_for_backward(y)
        return y

    @staticmethod
    def backward(ctx, dy):
        return dy * 2.0, None


def test_plain_tensors_take_the_forward_alone():
    x = torch.randn(3)
    assert ops._apply(_Twice, x).grad_fn is None
    assert ops._apply(_Twice, x.requires_grad_()).grad_fn is not None
    with torch.no_grad():
        assert ops._apply(_Twice, x).grad_fn is None


@pytest.mark.parametrize("grad", [True, False])
def test_a_tangent_is_not_dropped(grad):
    """Forward mode: refused, as by ``apply`` of a function without a jvp rule."""
    with torch.set_grad_enabled(grad), fwAD.dual_level():
        x = fwAD.make_dual(torch.randn(3), torch.ones(3))
        with pytest.raises(RuntimeError, match="(?i)forward|jvp"):
            ops._apply(_Twice, x)


def test_function_transforms_are_refused():
    for f in (lambda t: torch.func.vmap(lambda x: ops._apply(_Twice, x))(t),
              lambda t: torch.func.jvp(lambda x: ops._apply(_Twice, x), (t,), (torch.ones_like(t),))):
        with pytest.raises(RuntimeError):
            f(torch.randn(3, 4))
