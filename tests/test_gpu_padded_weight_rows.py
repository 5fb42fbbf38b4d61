"""dgrad on the row-wise weight codes where a matrix's rows are no whole number of K steps: the copy holds zero rows up to the
next multiple of 128 and the forward GEMM steps over them.  Bit for bit the outputs and gradients of the route through a
transposed copy of the codes, at widths around the K step, the 128-element tile and the GEMM tiles, dense and grouped (short,
empty and single-row groups), on tiles of every size the sizes pick, and with an expert whose weight holds infinities and NaN
next to experts without."""

import pytest
import torch

pytestmark = pytest.mark.gpu

WIDTHS = [(32, 32), (96, 160), (288, 64), (416, 288), (128, 992), (1056, 544), (992, 2080)]


def _config(recipe):
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    if recipe == "mxfp4":
        return Float4QuantConfig(activation_format=Format.E2M1_X2)
    if recipe == "tensorwise":
        return Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)
    return Float8QuantConfig(format=Format.E4M3, granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)


def _both_routes(step):
    import primus_amd.pytorch as turbo

    outs = []
    try:
        for flag in (True, False):
            turbo.ops.set_dgrad_reads_rowwise_weight(flag)
            outs.append(step(turbo.ops))
    finally:
        turbo.ops.set_dgrad_reads_rowwise_weight(True)
    for i, (got, want) in enumerate(zip(*outs)):
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (i, got, want)


@pytest.mark.parametrize("lens", [None, [70, 0, 1, 300, 129]])
@pytest.mark.parametrize("n,k", WIDTHS)
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "tensorwise"])
def test_gradients_do_not_depend_on_the_route(gpu, recipe, n, k, lens):
    cfg, m = _config(recipe), 333 if lens is None else sum(lens)
    gen = torch.Generator().manual_seed(n + k)
    x0 = torch.randn(m, k, generator=gen).bfloat16().to(gpu)
    w0 = (torch.randn(*(() if lens is None else (len(lens),)), n, k, generator=gen) * 0.05).bfloat16().to(gpu)
    dy = torch.randn(m, n, generator=gen).bfloat16().to(gpu)
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)

    def step(ops):
        x, w = x0.clone().requires_grad_(), w0.clone().requires_grad_()
        if lens is None:
            y = (ops.gemm_fp4 if recipe == "mxfp4" else ops.gemm_fp8)(x, w, trans_b=True, config=cfg)
        else:
            y = (ops.grouped_gemm_fp4 if recipe == "mxfp4" else ops.grouped_gemm_fp8)(x, w, gl, trans_b=True, config=cfg)
        return (y, *torch.autograd.grad(y, (x, w), dy))

    _both_routes(step)


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4"])
def test_formed_inputs_and_a_bad_expert(gpu, recipe):
    cfg, lens, n, k = _config(recipe), [130, 40, 0, 257], 160, 96
    gen = torch.Generator().manual_seed(5)
    h0 = torch.randn(sum(lens), 2 * k, generator=gen).bfloat16().to(gpu)
    w0 = (torch.randn(4, n, k, generator=gen) * 0.05).bfloat16()
    w0[1, 0, :7], w0[1, 5, 3], w0[3, 2, 1] = float("inf"), float("nan"), float("nan")
    w0 = w0.to(gpu)
    probs = torch.rand(sum(lens), generator=gen).to(gpu)
    dy = torch.randn(sum(lens), n, generator=gen).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)

    def step(ops):
        h, w, p = h0.clone().requires_grad_(), w0.clone().requires_grad_(), probs.clone().requires_grad_()
        glu = ops.glu_grouped_gemm_fp4 if recipe == "mxfp4" else ops.glu_grouped_gemm_fp8
        y = glu(h, p, w, gl, activation="silu", trans_b=True, config=cfg)
        dh, dw, dp = torch.autograd.grad(y, (h, w, p), dy)
        assert dh[:130].isfinite().all()         # the first expert's weight is finite, its neighbour's is not
        return y, dh, dw, dp

    _both_routes(step)


def test_norm_in_front(gpu):
    cfg, m, n, k = _config("mxfp8"), 200, 352, 736
    gen = torch.Generator().manual_seed(6)
    x0 = torch.randn(m, k, generator=gen).bfloat16().to(gpu)
    w0 = (torch.randn(n, k, generator=gen) * 0.05).bfloat16().to(gpu)
    nw0 = torch.rand(k, generator=gen).bfloat16().to(gpu)
    dy = torch.randn(m, n, generator=gen).bfloat16().to(gpu)

    def step(ops):
        x, w, nw = x0.clone().requires_grad_(), w0.clone().requires_grad_(), nw0.clone().requires_grad_()
        y = ops.rmsnorm_gemm_fp8(x, nw, 1e-5, w, config=cfg)
        return (y, *torch.autograd.grad(y, (x, w, nw), dy))

    _both_routes(step)
