"""Which cached weight copies go to the linear's two native calls, which are told sizes and format and trust them: those
whose codes and scales are what the call's sizes and format describe.  Every other copy takes the launch-by-launch route,
whose GEMM wrappers take the format from the codes and check every shape, the device and the strides."""

import pytest
import torch

from primus_amd import _lib
from primus_amd.pytorch import kernels as K
from primus_amd.pytorch import ops
from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, QuantizedTensor, QuantizedTensorPair, ScaleDtype, ScalingGranularity

N, K_, ROWS = 64, 96, 8
FP8 = Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
FP4W = Float4QuantConfig(activation_format=Format.E4M3)


class _OnDevice(torch.Tensor):
    """A host tensor that says it is on the GPU: the routes are told apart before anything is launched."""

    is_cuda = property(lambda self: True)

    @property
    def device(self):
        return torch.device("cuda", 0)

    def get_device(self):
        return 0

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        with torch._C.DisableTorchFunctionSubclass():
            return func(*args, **(kwargs or {}))


def _gpu(t):
    return t.as_subclass(_OnDevice)


def _copy(rows, ld, fmt=_lib.FMT_E4M3, axis=-1, shape=None, layout=K.LAYOUT_KSTEP, code_rows=None, panels=None, wrap=_gpu, strided=False):
    """A cached copy of a weight with `rows` rows of `ld` elements, K-step-major."""
    ld_p = (ld + 127) // 128 * 128
    per = 2 if fmt == _lib.FMT_E2M1 else 1
    cs = K._code_shape(code_rows or rows, ld_p, per, layout)
    codes = torch.zeros(cs, dtype=torch.uint8).view(K._code_dtype(fmt))
    if strided:
        codes = torch.zeros(cs[:-1] + (2 * cs[-1],), dtype=torch.uint8)[..., :cs[-1]].view(K._code_dtype(fmt))
    ss = K._scale_shape(rows, ld_p, layout)
    scales = torch.zeros((panels or ss[0],) + tuple(ss[1:]), dtype=torch.uint8)
    return QuantizedTensor(wrap(codes), wrap(scales), logical_shape=shape or (rows, ld), axis=axis, use_2d_block=True, kchunk=layout)


class _Taken(Exception):
    pass


def _route(monkeypatch, weight, config, needs_grad=False):
    def stop(name):
        def f(*args, **kw):
            raise _Taken(name)
        return f

    monkeypatch.setattr(K, "linear_forward_impl", stop("two calls"))
    monkeypatch.setattr(K, "linear_plan", lambda *a, **kw: None)
    monkeypatch.setattr(K, "quantize_mx_impl", stop("launch by launch"))
    x = _gpu(torch.zeros(ROWS, K_, dtype=torch.bfloat16)).requires_grad_(needs_grad)
    op = ops.gemm_fp4 if isinstance(config, Float4QuantConfig) else ops.gemm_fp8
    with pytest.raises(_Taken) as taken:
        op(x, weight, config=config)
    return str(taken.value)


def test_a_matching_copy_takes_the_two_calls(monkeypatch):
    assert _route(monkeypatch, _copy(N, K_), FP8) == "two calls"
    assert _route(monkeypatch, _copy(N, K_, _lib.FMT_E2M1), FP4W) == "two calls"
    pair = QuantizedTensorPair(_copy(N, K_), _copy(K_, N, axis=-2))
    assert _route(monkeypatch, pair, FP8, needs_grad=True) == "two calls"


@pytest.mark.parametrize("fmt,config", [(_lib.FMT_E2M1, FP8), (_lib.FMT_E4M3, FP4W)], ids=["e2m1_in_fp8", "e4m3_in_fp4"])
def test_a_bare_copy_of_another_format(monkeypatch, fmt, config):
    assert _route(monkeypatch, _copy(N, K_, fmt), config) == "launch by launch"


@pytest.mark.parametrize("kw", [dict(code_rows=N - 32), dict(panels=2), dict(wrap=lambda t: t), dict(strided=True)],
                         ids=["rows", "panels", "host", "strided"])
def test_a_payload_the_sizes_do_not_describe(monkeypatch, kw):
    assert _route(monkeypatch, _copy(N, K_, **kw), FP8) == "launch by launch"


@pytest.mark.parametrize("kw", [dict(fmt=_lib.FMT_E2M1), dict(code_rows=K_ - 32), dict(wrap=lambda t: t), dict(strided=True), dict(rows=K_ + 32)],
                         ids=["format", "rows", "host", "strided", "size"])
def test_a_transposed_copy_that_does_not_match(monkeypatch, kw):
    data_t = _copy(**{"rows": K_, "ld": N, "axis": -2, **kw})
    assert _route(monkeypatch, QuantizedTensorPair(_copy(N, K_), data_t), FP8, needs_grad=True) == "launch by launch"
