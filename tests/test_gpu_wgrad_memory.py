"""The weight gradient on the side stream: passes that the host issues far ahead of the device need the memory of one, and what they
reuse in between holds the bits of one stream, in two calls and launch by launch."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu

PASSES = 8


def _linear(gpu, recipe, accumulate):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    cfg = {"mxfp8": Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
           "mxfp4": Float4QuantConfig(activation_format=Format.E2M1_X2),
           "tensorwise": Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)}[recipe]
    op = pt.ops.grouped_gemm_fp4 if recipe == "mxfp4" else pt.ops.grouped_gemm_fp8
    lens, n, k = [700, 0, 1, 835], 1056, 2080
    g = torch.Generator(device=gpu).manual_seed(7)
    xs = [torch.randn(sum(lens), k, generator=g, device=gpu).bfloat16().requires_grad_() for _ in range(PASSES)]
    dys = [torch.randn(sum(lens), n, generator=g, device=gpu).bfloat16() for _ in range(PASSES)]
    w = (torch.randn(len(lens), n, k, generator=g, device=gpu) * 0.05).bfloat16().requires_grad_()
    if accumulate:
        w.main_grad = torch.zeros(w.shape, device=gpu)
        w.grad_added_to_main_grad = False
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)

    def run(i):
        y = op(xs[i], w, gl, trans_b=True, config=cfg, fuse_bgrad_accum_pattern="megatron" if accumulate else None)
        return torch.autograd.grad(y, (xs[i], w), dys[i])

    return run, w


@contextlib.contextmanager
def _route(observed):
    from primus_amd.pytorch import kernels as K

    K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
    try:
        yield
    finally:
        K.set_launch_hook(None)


@pytest.mark.parametrize("observed", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "tensorwise"])
def test_passes_issued_ahead(gpu, recipe, accumulate, observed, monkeypatch):
    from primus_amd.pytorch import ops

    monkeypatch.setattr(ops, "_overlaps", lambda plan: True)
    run, w = _linear(gpu, recipe, accumulate)
    busy = torch.randn(8192, 8192, device=gpu, dtype=torch.bfloat16)
    there = torch.cuda.Event()

    def passes():
        out, held = [], []
        for i in range(PASSES):
            g = run(i)
            if i % 2:
                out += [t.clone() for t in g[: 1 if accumulate else 2]]
            del g
            held.append(torch.cuda.memory_stats()["active_bytes.all.current"] - sum(t.nbytes for t in out))
        if accumulate:
            out.append(w.main_grad.clone())
            w.main_grad.zero_()
        return out, held

    with _route(observed):
        monkeypatch.setattr(ops, "_wgrad_overlap", False)
        want, _ = passes()
        monkeypatch.setattr(ops, "_wgrad_overlap", True)
        passes()
        torch.cuda.synchronize()
        for _ in range(100):
            torch.mm(busy, busy)      # nothing below starts while the host issues it
        there.record()
        got, held = passes()
        assert not there.query()
    assert max(held) - held[0] < 1 << 20, held
    for a, b in zip(want, got):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
