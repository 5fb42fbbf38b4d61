"""A linear of the 128-blockwise recipe in two calls (one quantiser launch per direction) against the launch-by-launch route
that a launch observer selects: the same bits, with either gradient left out, ragged and empty groups, an accumulated main_grad,
and sizes around the tiles and the 4 x 4 supertiles of the quantiser's launch."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(x, w, gl, dy, wrt, accum):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch.core import Float8QuantConfig, Format, ScalingGranularity

    cfg = Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.BLOCKWISE, block_size=128)
    kw = {"fuse_bgrad_accum_pattern": "megatron"} if accum else {}
    if gl is None:
        y = pt.ops.gemm_fp8(x, w, trans_a=False, trans_b=True, out_dtype=None, config=cfg, **kw)
    else:
        y = pt.ops.grouped_gemm_fp8(x, w, gl, trans_b=True, config=cfg, **kw)
    grads = torch.autograd.grad(y, wrt, dy) if wrt else ()
    return (y.detach(),) + (grads if not accum else grads[:1])


@pytest.mark.parametrize("lens,rows,n,k", [(None, 1, 128, 128), (None, 200, 640, 384), (None, 700, 256, 1152), ([0, 130, 1, 0, 300, 64], 495, 256, 640),
                                           ([7, 0], 7, 128, 256)])
@pytest.mark.parametrize("needs", ["both", "input", "weight", "none", "main_grad"])
def test_two_calls_give_the_same_bits(gpu, lens, rows, n, k, needs):
    from primus_amd.pytorch import kernels as K

    g = torch.Generator().manual_seed(rows + n + k)
    x = torch.randn(rows, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(*(() if lens is None else (len(lens),)), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    x[0, 3] = float("inf")
    dy = torch.randn(rows, n, generator=g).bfloat16().to(gpu)
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    x.requires_grad_(needs in ("both", "input", "main_grad"))
    w.requires_grad_(needs in ("both", "weight", "main_grad"))
    wrt = [t for t in (x, w) if t.requires_grad]
    accum = needs == "main_grad"
    out = []
    for observed in (True, False):
        if accum:
            w.main_grad = torch.ones_like(w, dtype=torch.float32)
            w.grad_added_to_main_grad = False
        K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
        try:
            got = _step(x, w, gl, dy, wrt, accum)
        finally:
            K.set_launch_hook(None)
        if accum:
            assert w.grad_added_to_main_grad
            got += (w.main_grad,)
        out.append([t.clone() for t in got])
    for a, b in zip(*out):
        assert a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8))
