"""Experts bound by their weights (more than 256 MiB of codes, under 512 rows per group), whose backward runs the weight gradient in front
of dgrad: the bits of the launch-by-launch route, which runs dgrad first; also where only one of the two is asked for, with an
activation in front, and with the weight gradient added to a float32 buffer.  A dgrad that is refused leaves that buffer alone."""

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


@pytest.mark.parametrize("activation", ["silu", "gelu"])
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4"])
def test_with_an_activation_in_front_and_a_main_grad(gpu, recipe, activation):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    cfg = {"mxfp8": Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
           "mxfp4": Float4QuantConfig(activation_format=Format.E2M1_X2)}[recipe]
    fused = pt.ops.glu_grouped_gemm_fp8 if recipe == "mxfp8" else pt.ops.glu_grouped_gemm_fp4
    lens, (n, f) = [0, 1, 130, 700], ((8352, 8192) if recipe == "mxfp8" else (16544, 8192))
    gen = torch.Generator(device=gpu).manual_seed(n)
    rows = sum(lens)
    h, dy = (torch.randn(rows, c, generator=gen, device=gpu).bfloat16() for c in (2 * f, n))
    probs = torch.rand(rows, generator=gen, device=gpu)
    mask = torch.arange(rows, device=gpu) % 7 != 3
    w = (torch.randn(len(lens), n, f, generator=gen, device=gpu, dtype=torch.bfloat16) * 0.05).requires_grad_()
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    h.requires_grad_()
    probs.requires_grad_()
    out = []
    for accumulate in (None, "megatron"):
        for observed in (True, False):
            w.grad_added_to_main_grad = False
            w.main_grad = torch.ones(w.shape, device=gpu) if accumulate else None
            K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
            try:
                y = fused(h, probs, w, gl, activation=activation, row_mask=mask, config=cfg, fuse_bgrad_accum_pattern=accumulate)
                got = torch.autograd.grad(y, (h, probs, w), dy)
            finally:
                K.set_launch_hook(None)
            out.append((y.detach(), got[0], got[1], w.main_grad if accumulate else got[2]))
        for a, b in zip(*out):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        out.clear()


@pytest.mark.parametrize("fmt,n,k", [(0, 8352, 8192), (1, 16544, 8192)])
def test_a_refused_dgrad_adds_nothing_to_the_weight_gradient(gpu, fmt, n, k):
    from primus_amd import _lib
    from primus_amd.pytorch import kernels as K

    lens = [0, 1, 130, 700]
    rows = sum(lens)
    x, dy = (torch.ones(rows, c, device=gpu, dtype=torch.bfloat16) for c in (k, n))
    w = torch.ones(len(lens), n, k, device=gpu, dtype=torch.bfloat16)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    plan = K.linear_plan(rows, n, k, len(lens), _lib.LINEAR_MX, fmt, fmt, fmt, 0, True, True, True)
    _, saved = K.linear_forward_impl(plan, x, w, None, gl)
    scratch = torch.empty(plan.bwd_bytes, dtype=torch.uint8, device=gpu)
    dw = torch.zeros(len(lens), n, k, device=gpu)
    with pytest.raises(_lib.MXLinearError):
        K.linear_backward_impl(plan, _lib.LINEAR_QUANTIZE | _lib.LINEAR_DX | _lib.LINEAR_DW, dy, saved, scratch, None, dw, group_lens=gl, accumulate=True)
    assert not dw.any()
