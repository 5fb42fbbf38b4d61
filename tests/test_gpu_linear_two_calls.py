"""A linear issued in two calls (mxl_linear_forward / mxl_linear_backward) against the launch-by-launch route of the same
operators, which a launch observer selects: the same kernels on the same buffers' contents, so the same bits."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


def _launch_by_launch(fn):
    from primus_amd.pytorch import kernels as K

    K.set_launch_hook(lambda name, info: contextlib.nullcontext())
    try:
        return fn()
    finally:
        K.set_launch_hook(None)


def _config(recipe):
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    if recipe == "tensorwise":
        return Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)
    if recipe == "mxfp8":
        return Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
    if recipe == "mxfp4w8":
        return Float4QuantConfig(activation_format=Format.E4M3)
    return Float4QuantConfig(use_gradient_sr=True, colwise_rht_signs=0xA6C9)


def _check(run, leaves):
    from primus_amd.pytorch import ops

    def step():
        ops.manual_sr_seed(11)
        y = run()
        dy = torch.linspace(-2, 2, y.numel(), device=y.device).view_as(y).bfloat16()
        with torch.no_grad():
            y0 = run()
        return (y, y0) + torch.autograd.grad(y, leaves, dy)

    rule = ops._overlaps
    try:
        want = _launch_by_launch(step)
        for together in (True, False):     # the weight gradient on the side stream, and everything in one call
            ops._overlaps = lambda plan: together
            got = step()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))
        assert torch.equal(want[0], want[1])
    finally:
        ops._overlaps = rule
        ops.manual_sr_seed(None)


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4", "tensorwise"])
@pytest.mark.parametrize("lens,n,k", [(None, 96, 160), (None, 256, 384), ([33, 0, 130, 1, 92], 160, 96), ([300, 212], 384, 512)])
def test_plain_linear(gpu, recipe, lens, n, k):
    from primus_amd.pytorch import ops

    m = 71 if lens is None else sum(lens)
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(*(() if lens is None else (len(lens),)), n, k, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    cfg = _config(recipe)
    fp4 = recipe.startswith("mxfp4")
    if lens is None:
        op = ops.gemm_fp4 if fp4 else ops.gemm_fp8
        run = lambda: op(x, w, config=cfg)  # noqa: E731
    else:
        op = ops.grouped_gemm_fp4 if fp4 else ops.grouped_gemm_fp8
        run = lambda: op(x, w, gl, config=cfg)  # noqa: E731
    _check(run, [x, w])
    _check(run, [x])
    _check(run, [w])


@pytest.mark.parametrize("kind", ["silu", "gelu", "norm"])
def test_fused_inputs(gpu, kind):
    from primus_amd.pytorch import ops

    g = torch.Generator().manual_seed(5)
    cfg = _config("mxfp8")
    if kind == "norm":
        x = torch.randn(131, 288, generator=g).bfloat16().to(gpu).requires_grad_()
        nw = torch.randn(288, generator=g).bfloat16().to(gpu).requires_grad_()
        w = (torch.randn(96, 288, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
        _check(lambda: ops.rmsnorm_gemm_fp8(x, nw, 1e-5, w, config=cfg), [x, nw, w])
        return
    lens = [33, 0, 130, 1, 92]
    m = sum(lens)
    x = torch.randn(m, 2 * 160, generator=g).bfloat16().to(gpu).requires_grad_()
    probs = torch.rand(m, generator=g).to(gpu).requires_grad_()
    mask = (torch.arange(m) % 7 != 3).to(gpu)
    w = (torch.randn(len(lens), 128, 160, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    _check(lambda: ops.glu_grouped_gemm_fp8(x, probs, w, gl, activation=kind, row_mask=mask, config=cfg), [x, probs, w])


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4"])
def test_cached_weights(gpu, recipe):
    from primus_amd.pytorch import ops
    from primus_amd.pytorch.core import QuantizedTensorPair, create_quantized_weight, float4_e2m1fn_x2, float8_e4m3

    lens, n, k = [33, 0, 130, 1, 92], 160, 96
    g = torch.Generator().manual_seed(9)
    x = torch.randn(sum(lens), k, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(len(lens), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    cfg = _config(recipe)
    pair = QuantizedTensorPair(*create_quantized_weight(w, float8_e4m3 if recipe == "mxfp8" else float4_e2m1fn_x2, cfg))
    op = ops.grouped_gemm_fp8 if recipe == "mxfp8" else ops.grouped_gemm_fp4
    _check(lambda: op(x, pair, gl, config=cfg), [x])


def test_accumulating_weight_gradient(gpu):
    from primus_amd.pytorch import ops

    g = torch.Generator().manual_seed(3)
    x = torch.randn(200, 256, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(128, 256, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    w.grad_added_to_main_grad = False

    def step():
        w.main_grad = torch.ones(128, 256, device=gpu)
        y = ops.gemm_fp8(x, w, config=_config("mxfp8"), fuse_bgrad_accum_pattern="megatron")
        dx, _ = torch.autograd.grad(y, [x, w], torch.ones_like(y))
        return dx, w.main_grad

    want = _launch_by_launch(step)
    assert all(torch.equal(a, b) for a, b in zip(step(), want))


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("shape,n", [((3, 100, 256), 192), ((71, 160), 96)])
def test_local_mxfp4_linear_and_its_function(gpu, sr, shape, n):
    """``mxfp4_linear`` in eager mode runs on the operators; output and both gradients have the bits of
    ``MXFP4LinearFunction``, which serves everything else, in either byte order."""
    from primus_amd.megatron.extensions.primus_turbo_mxfp4_local import MXFP4LinearFunction, mxfp4_linear
    from primus_amd.pytorch import ops

    g = torch.Generator().manual_seed(n)
    x = torch.randn(*shape, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(n, shape[-1], generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    dy = torch.randn(*shape[:-1], n, generator=g).bfloat16().to(gpu)

    def step(linear):
        ops.manual_sr_seed(23)
        y = linear()
        return (y,) + torch.autograd.grad(y, [x, w], dy)

    try:
        got = step(lambda: mxfp4_linear(x, w, use_gradient_sr=sr))
        for pre in (False, True):
            want = step(lambda: MXFP4LinearFunction.apply(x, w, pre, False, None, 0, 0, sr)[0])
            assert all(torch.equal(a, b) for a, b in zip(got, want)), pre
    finally:
        ops.manual_sr_seed(None)
