"""A linear's two gradients in one launch against the launch-by-launch route (which a launch observer selects): the same
tiles, so the same bits.  One size per kernel of the pair: 64 x 128 or 128 x 128 tiles for the input gradient, two or
four stages for the weight gradient, the weight's own codes (sizes in multiples of 128) or the transposed copy; and
sizes where only one of the two runs on small tiles."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


def _config(recipe):
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    if recipe == "tensorwise":
        return Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)
    if recipe == "mxfp8":
        return Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
    return Float4QuantConfig()


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "tensorwise"])
@pytest.mark.parametrize("m,n,k", [
    (257, 256, 384), (257, 160, 352),            # 64 x 128 tiles, two stages
    (1100, 256, 384), (1100, 160, 352),          # 64 x 128 tiles, four stages
    (1000, 256, 2944), (1000, 160, 2880),        # 128 x 128 tiles, two stages
    (1100, 256, 2944), (1100, 160, 2880),        # 128 x 128 tiles, four stages
    (64, 8192, 4096),                            # the weight gradient's 512 tiles of 256 x 256 against few rows
    (4096, 128, 4096),                           # the input gradient on 256 x 256 tiles
])
def test_gradients_in_one_launch(gpu, recipe, m, n, k):
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(n, k, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    dy = torch.randn(m, n, generator=g).bfloat16().to(gpu)
    op = ops.gemm_fp4 if recipe == "mxfp4" else ops.gemm_fp8

    def step():
        return torch.autograd.grad(op(x, w, config=_config(recipe)), [x, w], dy)

    got = step()
    K.set_launch_hook(lambda name, info: contextlib.nullcontext())
    try:
        want = step()
    finally:
        K.set_launch_hook(None)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
