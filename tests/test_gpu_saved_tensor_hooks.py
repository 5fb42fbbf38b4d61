"""A linear's backward under saved-tensor hooks: tensors that went through host memory give the same gradients, tensors that
come back with other strides are refused."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(recipe, gpu):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch.core import Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    g = torch.Generator().manual_seed(7)
    x = torch.randn(200, 256, generator=g).bfloat16().to(gpu).requires_grad_()
    w = (torch.randn(384, 256, generator=g) * 0.05).bfloat16().to(gpu).requires_grad_()
    nw = torch.rand(256, generator=g).bfloat16().to(gpu).requires_grad_()
    dy = torch.randn(200, 384, generator=g).bfloat16().to(gpu)
    mx = Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
    if recipe == "norm":
        return (lambda: pt.ops.rmsnorm_gemm_fp8(x, nw, 1e-5, w, config=mx)), [x, nw, w], dy
    cfg = {"mxfp8": mx, "tensorwise": Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE),
           "blockwise": Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.BLOCKWISE, block_size=128)}[recipe]
    return (lambda: pt.ops.gemm_fp8(x, w, config=cfg)), [x, w], dy


@pytest.mark.parametrize("recipe", ["mxfp8", "tensorwise", "blockwise", "norm"])
def test_through_host_memory(gpu, recipe):
    run, leaves, dy = _run(recipe, gpu)
    want = torch.autograd.grad(run(), leaves, dy)
    with torch.autograd.graph.save_on_cpu():
        y = run()
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, leaves, dy), want))


@pytest.mark.parametrize("recipe", ["blockwise", "norm"])
def test_other_strides_are_refused(gpu, recipe):
    run, leaves, dy = _run(recipe, gpu)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.t().contiguous(), lambda t: t.t()):
        y = run()
    with pytest.raises(ValueError, match="contiguous"):
        torch.autograd.grad(y, leaves, dy)
