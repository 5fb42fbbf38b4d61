"""A float32 ``main_grad`` that is not on the gradient's device is refused before the GEMM is handed its address."""

import types

import pytest
import torch

from primus_amd.pytorch import kernels as K
from primus_amd.pytorch import ops

PLAN = types.SimpleNamespace(bwd_bytes=16, rows=4, n=32, k=64, groups=0)


def _backward(target):
    owner = types.SimpleNamespace(dtype=torch.bfloat16, grad_added_to_main_grad=False)
    return ops._backward_in_parts(PLAN, torch.zeros(4, 32, dtype=torch.bfloat16), None, None, (target, owner), False, True, (32, 64), None)


def test_a_buffer_on_another_device_is_refused(monkeypatch):
    calls = []
    monkeypatch.setattr(K, "linear_backward_impl", lambda *a, **kw: calls.append(a))
    with pytest.raises(ValueError, match="device"):
        _backward(torch.zeros(32, 64, device="meta"))
    assert not calls
    _backward(torch.zeros(32, 64))
    assert len(calls) == 1
