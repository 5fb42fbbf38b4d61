"""``mxfp4_linear`` outside plain eager calls: function transforms and fake tensors go through ``MXFP4LinearFunction``,
which has a ``setup_context`` and custom ops with fake kernels for them."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from primus_amd.megatron.extensions import primus_turbo_mxfp4_local as local
from primus_amd.pytorch import ops

M, N, K = 32, 64, 96


@pytest.fixture
def on_the_host(monkeypatch):
    """The function's custom ops with host stand-ins: zero codes, and products that are all ones."""
    def dual(*args):
        return tuple(torch.zeros(t.shape, dtype=torch.uint8).view(t.dtype) for t in local._quantize_mxfp4_dual_fake(*args))

    def gemm(a, a_scale, b, b_scale, out_dtype, preshuffled):
        return torch.ones(a.shape[0], b.shape[0], dtype=out_dtype)

    monkeypatch.setattr(local, "_quantize_mxfp4_dual_op", dual)
    monkeypatch.setattr(local, "_gemm_fp4_nt_op", gemm)


def _operands():
    return torch.randn(M, K, dtype=torch.bfloat16), torch.randn(N, K, dtype=torch.bfloat16)


def test_plain_eager_calls_run_on_the_operators(monkeypatch):
    x, w = _operands()
    monkeypatch.setattr(ops, "mxfp4_linear_2d", lambda a, b, sr, signs: a.new_full((M, N), 3.0))
    assert local.mxfp4_linear(x, w).unique().tolist() == [3.0]
    assert local.mxfp4_linear(x, torch.nn.Parameter(w)).unique().tolist() == [3.0]


def test_function_transforms(on_the_host):
    x, w = _operands()
    g = torch.func.grad(lambda t: local.mxfp4_linear(t, w).float().sum())(x)
    assert torch.equal(g, torch.ones_like(x))
    y, back = torch.func.vjp(local.mxfp4_linear, x, w)
    assert torch.equal(y, torch.ones_like(y))
    assert [tuple(t.shape) for t in back(torch.ones_like(y))] == [(M, K), (N, K)]


def test_fake_tensors():
    with FakeTensorMode():
        x, w = _operands()
        y = local.mxfp4_linear(x, w)
        assert tuple(y.shape) == (M, N) and y.dtype == torch.bfloat16
    assert tuple(local.mxfp4_linear(x, w).shape) == (M, N)      # ... and outside of the mode that made them


def test_a_dispatch_mode_sees_the_custom_ops(on_the_host, monkeypatch):
    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    monkeypatch.setattr(ops, "mxfp4_linear_2d", lambda *a: pytest.fail("not the custom ops"))
    with Mode():
        assert local.mxfp4_linear(*_operands()).unique().tolist() == [1.0]


def test_a_gradient_of_another_output_only(on_the_host, monkeypatch):
    """The FP8 mode hands out its kept operands; where only they have a gradient, the linear's own is zero."""
    from primus_amd.pytorch.core.low_precision import ScalingGranularity, float8_e5m2

    monkeypatch.setattr(local, "_fp8_tw_backward_op", lambda g, x, w, fmt: (g.sum() * x, g.sum() * w))
    x, w = (t.requires_grad_() for t in _operands())
    out = local.MXFP4LinearFunction.apply(x, w, False, True, float8_e5m2, ScalingGranularity.TENSORWISE.value, 0, False)
    dx, dw = torch.autograd.grad(out[1].sum() + out[2].sum(), [x, w])
    assert torch.equal(dx, torch.zeros_like(x)) and torch.equal(dw, torch.zeros_like(w))
