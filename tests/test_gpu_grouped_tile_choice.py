"""Grouped forward and dgrad on either side of the lines by which a launch picks its output tile: the tile it picks gives the bits of
the ring kernel (each output element runs the same MFMAs in the same order).  Which tile that is, test_gemm_tile_choice.py says."""

import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


def _lens(groups, rows):
    """Uneven, some empty, ``rows`` per group on average."""
    lens = [(2 * rows * (i % 5)) // 4 for i in range(groups)]
    lens[-1] += groups * rows - sum(lens)
    return lens


# FP8: n 2560 with k 256 (40 MiB of codes), 1408 (220 MiB, a short contraction) and 3328 (520 MiB) is over 300 ring tiles in the forward,
# and with k 3328 in dgrad; n 256 with k 2560 (40 MiB) in dgrad alone
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "mxfp4w8"])
@pytest.mark.parametrize("n,k,rows", [(2560, 256, 32), (2560, 256, 33), (2560, 256, 97), (2560, 256, 192), (2560, 256, 193), (2560, 3328, 16), (2560, 3328, 17),
                                      (2560, 3328, 32), (2560, 3328, 33), (2560, 3328, 65), (2560, 1408, 32), (2560, 1408, 33),
                                      (256, 2560, 32), (256, 2560, 192), (256, 2560, 193)])
def test_the_tile_a_grouped_launch_picks(gpu, recipe, n, k, rows):
    from primus_amd.pytorch import kernels as K

    groups = 64
    lens = _lens(groups, rows)
    assert min(lens) >= 0 and sum(lens) == groups * rows
    afmt, wfmt, lay = {"mxfp8": (0, 0, 2), "mxfp4": (1, 1, 3), "mxfp4w8": (0, 1, 2)}[recipe]
    gen = torch.Generator(device=gpu).manual_seed(rows + k)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)

    def operand(shape):
        return torch.randn(shape, generator=gen, device=gpu, dtype=torch.bfloat16)

    xq = K.quantize_mx_impl(operand((sum(lens), k)), afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
    wq = K.quantize_mx_weight_2d_impl(operand((groups, n, k)), wfmt, rowwise=True, colwise=True, pad_to=128, kchunk=lay)
    runs = [lambda tile: K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=lay, tile=tile)]
    if afmt == wfmt:
        dq = K.quantize_mx_impl(operand((sum(lens), n)), afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
        runs.append(lambda tile: K.grouped_gemm_mx_nt_impl(dq[0], dq[1], wq[0], wq[3], gl, kchunk=lay, b_transposed=True, tile=tile))
    for run in runs:
        picked = run(None)
        assert torch.equal(picked.view(torch.int16), run("256").view(torch.int16))


# weights that the call quantises itself, 40 MiB of codes
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "mxfp4w8", "tensorwise"])
@pytest.mark.parametrize("rows", [32, 33, 64, 65, 128, 129, 192, 193])
def test_the_tile_behind_the_quantiser(gpu, recipe, rows):
    import primus_amd.pytorch as pt
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    cfg = {"mxfp8": Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
           "tensorwise": Float8QuantConfig(format=Format.HYBRID, granularity=ScalingGranularity.TENSORWISE),
           "mxfp4": Float4QuantConfig(activation_format=Format.E2M1_X2), "mxfp4w8": Float4QuantConfig(activation_format=Format.E4M3)}[recipe]
    op = pt.ops.grouped_gemm_fp4 if "fp4" in recipe else pt.ops.grouped_gemm_fp8
    groups, n, k = 64, 2560, 256
    lens = _lens(groups, rows)
    gen = torch.Generator(device=gpu).manual_seed(rows)
    x = torch.randn(groups * rows, k, generator=gen, device=gpu, dtype=torch.bfloat16)
    w = torch.randn(groups, n, k, generator=gen, device=gpu, dtype=torch.bfloat16) * 0.05
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    out = []
    for observed in (True, False):
        K.set_launch_hook((lambda name, info: contextlib.nullcontext()) if observed else None)
        try:
            with torch.no_grad():
                out.append(op(x, w, gl, trans_b=True, config=cfg))
        finally:
            K.set_launch_hook(None)
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
