"""Linears in two calls on both sides of the lines between codes stored through the caches and past them (a weight of 256 MiB of
codes and one just below, few rows and 512): the bits of the launch-by-launch route, which always streams them."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recipe", ["mxfp8", "blockwise"])
@pytest.mark.parametrize("rows,n,k", [(3, 16384, 16384), (3, 16256, 16384), (511, 16384, 16384), (512, 16384, 16384)])
def test_the_same_bits_either_way(gpu, recipe, rows, n, k):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch.core import Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    cfg = {"mxfp8": Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
           "blockwise": Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.BLOCKWISE, block_size=128)}[recipe]
    g = torch.Generator(device=gpu).manual_seed(rows)
    x, dy = (torch.randn(rows, c, generator=g, device=gpu).bfloat16() for c in (k, n))
    w = torch.randn(n, k, generator=g, device=gpu, dtype=torch.bfloat16) * 0.05
    x.requires_grad_()
    w.requires_grad_()
    out = []
    for observed in (True, False):
        K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
        try:
            y = pt.ops.gemm_fp8(x, w, trans_a=False, trans_b=True, out_dtype=None, config=cfg)
            out.append((y.detach(),) + torch.autograd.grad(y, (x, w), dy))
        finally:
            K.set_launch_hook(None)
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
