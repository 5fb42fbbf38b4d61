"""Linears in two calls on both sides of the lines between codes stored through the caches and past them (a weight of 256 MiB of
codes and one just below, few rows and 512), and in every other form with a row-wise copy that is kept and a transposed one that is not
(more than 64 MiB): the bits of the launch-by-launch route, which always streams them.  Small sizes, where both are kept, are
test_gpu_linear_two_calls'; weight-bound experts, where neither is, test_gpu_wgrad_first's."""

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


@pytest.mark.parametrize("form", ["mxfp4_sr_rht", "mxfp4_grouped", "mxfp8_grouped", "silu", "gelu_mxfp4", "norm"])
def test_one_copy_kept_and_one_not(gpu, form):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    ops, fp4 = pt.ops, "mxfp4" in form
    if form == "mxfp4_sr_rht":
        cfg = Float4QuantConfig(activation_format=Format.E2M1_X2, use_gradient_sr=True, colwise_rht_signs=0xA6C9)
    elif fp4:
        cfg = Float4QuantConfig(activation_format=Format.E2M1_X2)
    else:
        cfg = Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
    grouped = "grouped" in form or "lu" in form
    lens, n, k = [4100, 0, 1, 4111], 96, 16384 if fp4 else 8192
    m, g = sum(lens), torch.Generator(device=gpu).manual_seed(len(form))
    assert m * k // (2 if fp4 else 1) > 64 << 20 and m >= 512 * len(lens)
    x = torch.randn(m, 2 * k if "lu" in form else k, generator=g, device=gpu, dtype=torch.bfloat16)
    dy = torch.randn(m, n, generator=g, device=gpu, dtype=torch.bfloat16)
    w = torch.randn(*([len(lens)] if grouped else []), n, k, generator=g, device=gpu, dtype=torch.bfloat16) * 0.05
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    probs = torch.rand(m if "lu" in form else k, generator=g, device=gpu)
    leaves = [x, w]
    if "lu" in form:
        leaves.append(probs)
        op = ops.glu_grouped_gemm_fp4 if fp4 else ops.glu_grouped_gemm_fp8
        run = lambda: op(x, probs, w, gl, activation=form[:4], config=cfg)  # noqa: E731
    elif form == "norm":
        leaves.append(probs := probs.bfloat16())
        run = lambda: ops.rmsnorm_gemm_fp8(x, probs, 1e-5, w, config=cfg)  # noqa: E731
    elif grouped:
        op = ops.grouped_gemm_fp4 if fp4 else ops.grouped_gemm_fp8
        run = lambda: op(x, w, gl, trans_b=True, config=cfg)  # noqa: E731
    else:
        run = lambda: ops.gemm_fp4(x, w, trans_b=True, config=cfg)  # noqa: E731
    for t in leaves:
        t.requires_grad_()
    out = []
    try:
        for observed in (True, False):
            K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
            ops.manual_sr_seed(5)
            y = run()
            out.append((y.detach(),) + torch.autograd.grad(y, leaves, dy))
    finally:
        K.set_launch_hook(None)
        ops.manual_sr_seed(None)
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
