"""What autograd kept for a linear's backward in one call comes back through saved-tensor hooks: values with other strides, on
another device, of another type or length are refused before an address is handed to native code."""

import types

import pytest
import torch

from primus_amd import _lib
from primus_amd.pytorch import kernels as K

ROWS, N, K_, G = 40, 128, 256, 2
CODES = torch.float8_e4m3fn


def _zeros(nbytes, dtype=torch.uint8):
    return torch.zeros(nbytes, dtype=torch.uint8).view(dtype)


def _blockwise():
    plan = K.linear_plan(ROWS, N, K_, G, _lib.LINEAR_BLOCKWISE, _lib.FMT_E4M3, _lib.FMT_E4M3, _lib.FMT_E5M2, 0, True, True)
    return plan, {"x": torch.zeros(ROWS, K_).bfloat16(), "wt": torch.zeros(G, N, K_).bfloat16(), "group_lens": torch.tensor([30, 10])}


def _activation():
    plan = K.linear_plan(ROWS, N, K_, G, _lib.LINEAR_MX, _lib.FMT_E4M3, _lib.FMT_E4M3, _lib.FMT_E4M3, 0, True, True, True, False, _lib.LINEAR_SILU)
    return plan, {"saved": _zeros(plan.saved_bytes), "x": torch.zeros(ROWS, 2 * K_).bfloat16(), "group_lens": torch.tensor([30, 10]),
                  "aux0": torch.zeros(ROWS), "aux1": torch.zeros(ROWS, dtype=torch.uint8)}


def _norm():
    plan = K.linear_plan(ROWS, N, K_, 0, _lib.LINEAR_MX, _lib.FMT_E4M3, _lib.FMT_E4M3, _lib.FMT_E4M3, 0, True, True, True, False, _lib.LINEAR_RMSNORM)
    return plan, {"saved": _zeros(plan.saved_bytes), "x": torch.zeros(ROWS, K_).bfloat16(), "aux0": torch.zeros(K_).bfloat16()}


def _cached():
    plan = K.linear_plan(ROWS, N, K_, G, _lib.LINEAR_MX, _lib.FMT_E4M3, _lib.FMT_E4M3, _lib.FMT_E4M3, 0, True, False, False, True)
    return plan, {"wt": torch.zeros(N // 64, G * K_, 64).to(CODES), "wt_scales": torch.zeros(1, G * K_, 16, dtype=torch.uint8),
                  "group_lens": torch.tensor([30, 10])}


@pytest.fixture
def calls(monkeypatch):
    made = []
    for make in (_blockwise, _activation, _norm, _cached):
        make()                                   # (the plans' sizes come from the library)
    monkeypatch.setattr(_lib, "load", lambda: types.SimpleNamespace(mxl_linear_backward=lambda *a: made.append(a) or 0))
    monkeypatch.setattr(K, "_stream", lambda: 0)
    return made


def _run(plan, kept):
    kept = dict(kept)
    K.linear_backward_impl(plan, _lib.LINEAR_DX, None, kept.pop("saved", None), torch.empty(plan.bwd_bytes, dtype=torch.uint8), **kept)


def _spoiled(t):
    yield "strides", t.new_empty((*t.shape, 2))[..., 0]
    yield "device", t.to("meta")
    yield "length", t[1:] if t.dim() == 1 else t[:, 1:].contiguous()
    if t.dtype == torch.bfloat16:
        yield "type", t.half()


@pytest.mark.parametrize("make", [_blockwise, _activation, _norm, _cached])
def test_only_what_was_kept(calls, monkeypatch, make):
    monkeypatch.setattr(torch.Tensor, "get_device", lambda t: 0 if t.device.type == "cpu" else 1)
    plan, kept = make()
    _run(plan, kept)
    assert len(calls) == 1
    for name, t in kept.items():
        for what, bad in _spoiled(t):
            with pytest.raises(ValueError, match="kept"):
                _run(plan, {**kept, name: bad})
            assert len(calls) == 1, (name, what)
