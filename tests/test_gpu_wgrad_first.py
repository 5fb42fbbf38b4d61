"""Experts bound by their weights (more than 256 MiB of codes, under 512 rows per group), whose backward runs the weight gradient in front
of dgrad: the bits of the launch-by-launch route, which runs dgrad first; also where only one of the two is asked for."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4"])
@pytest.mark.parametrize("lens", [[0, 1, 130, 700], [3, 0, 0, 0]])
@pytest.mark.parametrize("wanted", [(True, True), (True, False), (False, True)])
def test_the_same_bits_in_either_order(gpu, recipe, lens, wanted):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    cfg = {"mxfp8": Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
           "mxfp4": Float4QuantConfig(activation_format=Format.E2M1_X2)}[recipe]
    gemm = pt.ops.grouped_gemm_fp8 if recipe == "mxfp8" else pt.ops.grouped_gemm_fp4
    n, k = (8352, 8192) if recipe == "mxfp8" else (16544, 8192)      # 261 and 259 MiB of codes
    gen = torch.Generator(device=gpu).manual_seed(len(lens))
    rows = sum(lens)
    x, dy = (torch.randn(rows, c, generator=gen, device=gpu).bfloat16() for c in (k, n))
    w = torch.randn(len(lens), n, k, generator=gen, device=gpu, dtype=torch.bfloat16) * 0.05
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    wrt = [t.requires_grad_() for t, want in zip((x, w), wanted) if want]
    out = []
    for observed in (True, False):
        K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
        try:
            y = gemm(x, w, gl, trans_b=True, config=cfg)
            out.append((y.detach(),) + torch.autograd.grad(y, wrt, dy))
        finally:
            K.set_launch_hook(None)
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
