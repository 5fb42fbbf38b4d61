"""The work a training program hands to the low-precision linear operators, as cases that can be timed and compared.

Four paths, all through the public operators of ``primus_amd.pytorch.ops`` (and the MXFP4 linear of the "local"
transformer spec):

``linear``       one dense linear, forward and backward on a bf16 weight, or forward only on the cached quantised copies
                 a program keeps between optimizer steps (evaluation, further microbatches)
``norm_linear``  the RMSNorm in front of a column-parallel linear, folded into the linear's quantiser
``local_fp4``    the MXFP4 linear of the local spec: Hadamard transform of the weight-gradient operands, optional
                 stochastic rounding of the gradients and pre-shuffled layouts
``experts``      the expert MLP of an MoE layer on permuted rows: fc1, gated SiLU with the router's probabilities, fc2;
                 ragged groups from a skewed router, tokens per expert on the device

and the recipes those paths are trained with: ``mxfp8``, ``mxfp4`` (every operand E2M1), ``mxfp4w8`` (E2M1 weights, E4M3
activations), ``tensorwise`` and ``blockwise`` (E4M3 forward, E5M2 gradients), ``bf16`` (outside the autocast).

A case holds ``path``, ``recipe``, ``tokens``, the linear's ``k`` and ``n`` or the experts' ``hidden`` and ``ffn``,
``experts`` and ``topk``, and the switches ``backward`` (input gradients are taken), ``cached`` (quantised weight copies
made beforehand; no weight gradient then), ``sr`` and ``preshuffle``.
"""

from __future__ import annotations

import math

import torch

import primus_amd.pytorch as pt
from primus_amd.megatron.extensions.primus_turbo_mxfp4_local import mxfp4_linear
from primus_amd.pytorch.core import (
    Float4QuantConfig,
    Float8QuantConfig,
    Format,
    QuantizedTensorPair,
    ScaleDtype,
    ScalingGranularity,
    create_quantized_weight,
    float4_e2m1fn_x2,
    float8_e4m3,
)

ops = pt.ops


def _linear(name, recipe, tokens, k, n, *, path="linear", backward=True, cached=False, sr=False, preshuffle=False):
    return {"name": name, "path": path, "recipe": recipe, "tokens": tokens, "k": k, "n": n, "backward": backward,
            "cached": cached, "sr": sr, "preshuffle": preshuffle}


def _experts(name, recipe, tokens, hidden, ffn, experts, topk, *, cached=False):
    return {"name": name, "path": "experts", "recipe": recipe, "tokens": tokens, "hidden": hidden, "ffn": ffn,
            "experts": experts, "topk": topk, "backward": True, "cached": cached}


def listed():
    return [
        # evaluation of a short batch through the up projection of a Llama-3-8B MLP: weights quantised once, no
        # gradients; one launch pair per call, so latency is what counts
        _linear("eval_mxfp8", "mxfp8", 64, 4096, 14336, backward=False, cached=True),
        # a short sequence through a 4096 x 4096 projection (the attention output), trained
        _linear("short_mxfp8", "mxfp8", 256, 4096, 4096),
        # GPT-OSS-120B sized linear on a token count that fits no tile: k not a multiple of 128
        _linear("ragged_mxfp8", "mxfp8", 1999, 2880, 5760),
        # the LayerNorm column-parallel linear of Llama-3-8B at its full microbatch of 8192 tokens
        _linear("norm_mxfp8", "mxfp8", 8192, 4096, 14336, path="norm_linear"),
        # the local spec's MXFP4 linear with stochastically rounded gradients
        _linear("local_mxfp4", "mxfp4", 4096, 4096, 14336, path="local_fp4", sr=True),
        # current scaling (the FP8 recipe most models start with), the down projection of the same MLP
        _linear("tensorwise", "tensorwise", 4096, 14336, 4096),
        # 128-blockwise scaling (the DeepSeek-V3 recipe) on one of its dense projections, ragged token count
        _linear("blockwise", "blockwise", 3000, 7168, 2048),
        # Mixtral-8x7B experts at the benchmark's size: the largest case
        _experts("experts_mixtral_mxfp8", "mxfp8", 16384, 4096, 14336, 8, 2),
        # a DeepSeek-V3 shard (32 of the experts) on a short microbatch: a few rows in most groups
        _experts("experts_deepseek_mxfp8", "mxfp8", 1024, 7168, 2048, 32, 8),
        # GPT-OSS-120B: 128 experts, E2M1 weights kept quantised, E4M3 activations, no weight gradient
        _experts("experts_gptoss_mxfp4w8", "mxfp4w8", 16384, 2880, 2880, 128, 4, cached=True),
        # the pure MXFP4 recipe on Mixtral experts, one quarter of the benchmark's tokens
        _experts("experts_mixtral_mxfp4", "mxfp4", 4096, 4096, 14336, 8, 2),
        # layers left outside the autocast: the bf16 grouped GEMM on the DeepSeek shard
        _experts("experts_deepseek_bf16", "bf16", 4096, 7168, 2048, 32, 8),
    ]


# matrix rate of a recipe relative to bf16, for the bound on a drawn case's cost
_SPEED = {"mxfp8": 2.0, "mxfp4": 3.0, "mxfp4w8": 2.0, "tensorwise": 2.0, "blockwise": 1.5, "bf16": 1.0}
_LARGEST = 6.0 * 32768 * 4096 * 3 * 14336 / 2.0     # the Mixtral case above


def _log(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def draw(rng):
    """Tokens over three decades (odd counts included), widths in multiples of 32 (128 where the recipe demands it)
    over the range from small proxies to the largest models above, every path, recipe and switch."""
    while True:
        path = rng.choice(["linear", "linear", "linear", "norm_linear", "local_fp4", "experts", "experts", "experts"])
        tokens = _log(rng, 16, 16384)
        if path == "experts":
            recipe = rng.choice(["mxfp8", "mxfp8", "mxfp4", "mxfp4w8", "tensorwise", "blockwise", "bf16"])
            m = 128 if recipe == "blockwise" else 32
            experts = rng.choice([8, 16, 32, 64, 128])
            case = _experts("", recipe, tokens, _log(rng, 1024, 7168, m), _log(rng, 1024, 14336, m), experts,
                            rng.choice([1, 2, 4, 8]), cached=recipe == "mxfp4w8")
            weights = 3.0 * experts * case["hidden"] * case["ffn"]
        else:
            recipe = {"norm_linear": "mxfp8", "local_fp4": "mxfp4"}.get(path) or rng.choice(["mxfp8", "mxfp8", "mxfp4", "tensorwise", "blockwise"])
            m = 128 if recipe == "blockwise" else 32
            cached = path == "linear" and recipe in ("mxfp8", "mxfp4") and rng.random() < 0.4
            case = _linear("", recipe, tokens, _log(rng, 512, 16384, m), _log(rng, 512, 16384, m), path=path,
                           backward=not cached, cached=cached, sr=path == "local_fp4" and rng.random() < 0.5,
                           preshuffle=path == "local_fp4" and rng.random() < 0.5)
            weights = float(case["k"] * case["n"])
        if weights <= 8 * 4096 * 3 * 14336 and work(case)["flops"] / _SPEED[recipe] <= _LARGEST:
            del case["name"]
            return case


def _config(recipe):
    if recipe == "mxfp8":
        return Float8QuantConfig(format=Format.E4M3, granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32)
    if recipe == "tensorwise":
        return Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE)
    if recipe == "blockwise":
        return Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.BLOCKWISE, block_size=128)
    if recipe in ("mxfp4", "mxfp4w8"):
        return Float4QuantConfig(activation_format=Format.E2M1_X2 if recipe == "mxfp4" else Format.E4M3)
    return None


def _normal(shape, gen, scale=1.0, outliers=False):
    x = torch.randn(shape, generator=gen, device=gen.device, dtype=torch.bfloat16)
    if outliers:    # 0.1 % of the entries times 50: what moves block scales and saturates codes
        x = torch.where(torch.rand(shape, generator=gen, device=gen.device) < 1e-3, x * 50.0, x)
    return x * scale if scale != 1.0 else x


def _weight(case, shape, gen, cfg):
    w = _normal(shape, gen, 0.02)
    if case["cached"]:
        dest = float4_e2m1fn_x2 if isinstance(cfg, Float4QuantConfig) else float8_e4m3
        return QuantizedTensorPair(*create_quantized_weight(w, dest, cfg))
    return w.requires_grad_(case["backward"])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cfg = _config(case["recipe"])
    state = {"case": case, "cfg": cfg, "seed": seed}
    grad = case["backward"]
    if case["path"] != "experts":
        k, n, rows = case["k"], case["n"], case["tokens"]
        state["x"] = _normal((rows, k), gen, outliers=True).requires_grad_(grad)
        state["w"] = _weight(case, (n, k), gen, cfg)
        if case["path"] == "norm_linear":
            state["norm_w"] = (1.0 + _normal((k,), gen, 0.1)).requires_grad_(grad)
        if grad:
            state["dy"] = _normal((rows, n), gen, 1e-3)
        return state
    hidden, ffn, experts, topk = case["hidden"], case["ffn"], case["experts"], case["topk"]
    rows = case["tokens"] * topk
    # a router that prefers some experts: Gaussian logits plus a bias per expert
    logits = torch.randn((case["tokens"], experts), generator=gen, device=gen.device)
    logits = logits + torch.randn((experts,), generator=gen, device=gen.device)
    top = torch.softmax(logits, dim=-1).topk(topk, dim=-1)
    idx = top.indices.reshape(-1)
    state["lens"] = torch.bincount(idx, minlength=experts)
    state["probs"] = top.values.reshape(-1)[torch.argsort(idx, stable=True)].contiguous().requires_grad_(grad)
    state["x"] = _normal((rows, hidden), gen).requires_grad_(grad)
    state["w1"] = _weight(case, (experts, 2 * ffn, hidden), gen, cfg)
    state["w2"] = _weight(case, (experts, hidden, ffn), gen, cfg)
    state["dy"] = _normal((rows, hidden), gen, 1e-3)
    return state


def _run_experts(s):
    cfg, lens = s["cfg"], s["lens"]
    recipe = s["case"]["recipe"]
    if recipe == "bf16":
        h = ops.grouped_gemm(s["x"], s["w1"], lens, trans_b=True)
    else:
        fc1 = ops.grouped_gemm_fp4 if isinstance(cfg, Float4QuantConfig) else ops.grouped_gemm_fp8
        h = fc1(s["x"], s["w1"], lens, trans_b=True, config=cfg)
    mask = ops.tokens_per_expert_to_mask(lens, h.shape[0])
    if recipe in ("mxfp8", "mxfp4", "mxfp4w8"):
        fc2 = ops.glu_grouped_gemm_fp4 if isinstance(cfg, Float4QuantConfig) else ops.glu_grouped_gemm_fp8
        return fc2(h, s["probs"], s["w2"], lens, activation="silu", row_mask=mask, trans_b=True, config=cfg)
    act = ops.swiglu_with_probs(h, s["probs"], mask)
    if recipe == "bf16":
        return ops.grouped_gemm(act, s["w2"], lens, trans_b=True)
    return ops.grouped_gemm_fp8(act, s["w2"], lens, trans_b=True, config=cfg)


def run(state):
    case, cfg = state["case"], state["cfg"]
    path = case["path"]
    if path == "experts":
        y = _run_experts(state)
        wrt = [state["x"], state["probs"]] + ([] if case["cached"] else [state["w1"], state["w2"]])
    elif path == "norm_linear":
        y = ops.rmsnorm_gemm_fp8(state["x"], state["norm_w"], 1e-5, state["w"], config=cfg)
        wrt = [state["x"], state["norm_w"], state["w"]]
    elif path == "local_fp4":
        if case["sr"]:
            ops.manual_sr_seed(state["seed"])       # a reproducible run restarts the rounding's random sequence
        y = mxfp4_linear(state["x"], state["w"], preshuffle=case["preshuffle"], use_gradient_sr=case["sr"])
        wrt = [state["x"], state["w"]]
    else:
        gemm = ops.gemm_fp4 if isinstance(cfg, Float4QuantConfig) else ops.gemm_fp8
        y = gemm(state["x"], state["w"], trans_a=False, trans_b=True, out_dtype=None, config=cfg)
        wrt = [state["x"], state["w"]]
    if not case["backward"]:
        return y
    return (y,) + torch.autograd.grad(y, wrt, state["dy"])


def work(case):
    """Each input read once and each output written once; 2 m n k for each matrix product of the pass."""
    cached = case["cached"]
    products = (2 if cached else 3) if case["backward"] else 1
    wbits = {"mxfp8": 8.25, "mxfp4": 4.25, "mxfp4w8": 4.25}.get(case["recipe"], 16) if cached else 16
    if case["path"] == "experts":
        rows, hidden, ffn = case["tokens"] * case["topk"], case["hidden"], case["ffn"]
        weights = case["experts"] * 3 * hidden * ffn
        flops = products * 2.0 * rows * 3 * hidden * ffn
        # x, dy read; y, dx written (bf16); probabilities read, their gradient written (fp32)
        bytes_ = rows * hidden * 8.0 + rows * 8.0 + 8.0 * case["experts"]
    else:
        rows, k, n = case["tokens"], case["k"], case["n"]
        weights = k * n
        flops = products * 2.0 * rows * k * n
        bytes_ = (rows * k + rows * n) * (4.0 if case["backward"] else 2.0)
        if case["path"] == "norm_linear":
            bytes_ += 4.0 * k
    bytes_ += weights * wbits / 8.0
    if cached and case["backward"]:
        bytes_ += weights * wbits / 8.0     # the transposed copies a cached pair holds for the input gradient
    elif case["backward"]:
        bytes_ += weights * 2.0             # weight gradients
    return {"bytes": float(bytes_), "flops": float(flops)}


def tolerance(case):
    """Codes and scales of every recipe are exact functions of the inputs, products accumulate in float32, and every
    output is rounded once to bf16: what two correct implementations may differ by is that rounding.  Against the same
    codes multiplied in 64 bits: 1.66e-3 for one linear under every recipe, 1.94e-3 for the experts, whose fc2 also
    quantises a bf16 fc1 output; four times that is stated."""
    return {"rel": 8e-3 if case["path"] == "experts" else 7e-3}
