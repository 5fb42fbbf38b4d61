"""abs-max of a tensor where its pieces meet: one element decides, at either end of a piece of 16384 values, of the last,
partly filled piece, of the tail of fewer than 8, and of what a workgroup reads in a second round (more than 512 pieces);
and the two tensors of a tensor-wise linear, whose maxima come from one launch."""

import pytest
import torch

pytestmark = pytest.mark.gpu
PIECE, WORKGROUPS = 16384, 512


@pytest.mark.parametrize("n", [9, PIECE - 1, PIECE, PIECE + 8, PIECE * WORKGROUPS + 9, PIECE * (WORKGROUPS + 1) + 16])
def test_one_element_decides(gpu, n):
    from primus_amd.pytorch import kernels as K

    x = torch.full((n,), 0.5, dtype=torch.bfloat16, device=gpu)
    for i in {0, 7, n // 8 * 8 - 1, n - 1, min(PIECE - 1, n - 1), min(PIECE, n - 1), n // 2}:
        x[i] = -3.0
        assert K.amax_impl(x).item() == 3.0, i
        x[i] = 0.5
    assert K.amax_impl(x).item() == 0.5


@pytest.mark.parametrize("m,k,n", [(1, 32, 32), (300, 4096, 64), (33, 64, 8192)])
def test_both_tensors_of_a_linear(gpu, m, k, n):
    """Each operand's scale is its own: scaling one of them by a power of two scales the output by it, bit for bit."""
    import primus_amd.pytorch as pt
    from primus_amd.pytorch.core import Float8QuantConfig, Format, ScalingGranularity

    cfg = Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)
    gen = torch.Generator().manual_seed(m + k + n)
    x = torch.randn(m, k, generator=gen).bfloat16().to(gpu)
    w = torch.randn(n, k, generator=gen).bfloat16().to(gpu)

    def run(a, b):
        return pt.ops.gemm_fp8(a, b, trans_a=False, trans_b=True, out_dtype=None, config=cfg)

    y = run(x, w)
    assert torch.equal(run(x * 64, w), y * 64)
    assert torch.equal(run(x, w / 256), y / 256)
