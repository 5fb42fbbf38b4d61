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


@pytest.mark.parametrize("f,rows", [(2560, 1152), (2560, 1153), (4096, 2048), (4096, 2049), (4104, 2048), (6656, 512), (6656, 513), (8192, 1024), (8192, 1025)])
def test_whatever_the_number_of_rows(gpu, f, rows):
    from primus_amd.pytorch import ops

    g = torch.Generator(device=gpu).manual_seed(f)
    x, dy = (torch.randn(rows, c, generator=g, device=gpu).bfloat16() for c in (2 * f, f))
    probs = torch.rand(rows, generator=g, device=gpu)
    out = []
    for some in (slice(None), slice(0, 500)):
        h, p = x[some].clone().requires_grad_(), probs[some].clone().requires_grad_()
        out.append([t[:500] for t in torch.autograd.grad(ops.swiglu_with_probs(h, p), (h, p), dy[some])])
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
