"""The probabilities' gradient is a float32 sum over a row, whose order is the row length's alone: the same bits from the fused operator and
the two it stands for, launch by launch and in two calls, with the weight gradient on the side stream and without -- at the row
lengths where the activation's workgroup changes its size, with part-filled passes of every size."""

import pytest
import torch

from tests import test_gpu_activation, test_gpu_linear_two_calls

pytestmark = pytest.mark.gpu

LENGTHS = [2528, 2560, 2912, 4352, 6624, 6656, 8224, 14336, 16416]


@pytest.mark.parametrize("together", [True, False])
@pytest.mark.parametrize("activation,fp4", [("silu", False), ("gelu", True)])
@pytest.mark.parametrize("f", LENGTHS)
def test_fused_and_in_two_operators(gpu, f, activation, fp4, together, monkeypatch):
    from primus_amd.pytorch import ops

    monkeypatch.setattr(ops, "_overlaps", lambda plan: together)
    test_gpu_activation.test_glu_grouped_gemm_equals_activation_then_grouped_gemm(gpu, activation, fp4, [33, 0, 70], f, 64)


@pytest.mark.parametrize("kind", ["silu", "gelu"])
@pytest.mark.parametrize("f", LENGTHS)
def test_two_calls_and_launch_by_launch(gpu, f, kind):
    from primus_amd.pytorch import ops

    g = torch.Generator().manual_seed(f)
    lens = [33, 0, 70]
    m = sum(lens)
    x = torch.randn(m, 2 * f, generator=g).bfloat16().to(gpu).requires_grad_()
    probs = torch.rand(m, generator=g).to(gpu).requires_grad_()
    mask = (torch.arange(m) % 7 != 3).to(gpu)
    w = (torch.randn(len(lens), 64, f, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    cfg = test_gpu_linear_two_calls._config("mxfp8")
    test_gpu_linear_two_calls._check(lambda: ops.glu_grouped_gemm_fp8(x, probs, w, gl, activation=kind, row_mask=mask, config=cfg), [x, probs, w])
