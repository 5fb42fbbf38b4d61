"""The small tiles with eight stages (one workgroup to a CU, contractions from 48 K steps on) against the ring kernel, bit for
bit: contractions on both sides of that line (contractions are multiples of 128, so 47 steps of 64 are 48, and 46 the last
number below it) and of a scale panel, more than 256 tiles, ragged rows and groups, transposed weight codes."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4"])
@pytest.mark.parametrize("tile", ["64", "64x128"])
@pytest.mark.parametrize("lens,n,steps", [(None, 128, 46), (None, 96, 47), (None, 256, 48), (None, 11296, 48), (None, 128, 53), (None, 160, 64), ([33, 0, 130, 1], 128, 50), ([0, 70], 96, 72)])
def test_eight_stages_give_the_same_bits(gpu, recipe, tile, lens, n, steps):
    from primus_amd.pytorch import kernels as K

    afmt, wfmt, lay = {"mxfp8": (0, 0, 2), "mxfp4w8": (0, 1, 2), "mxfp4": (1, 1, 3)}[recipe]
    k = (steps * (128 if afmt == 1 else 64) + 127) // 128 * 128
    m = 129 if lens is None else sum(lens)
    g = torch.Generator().manual_seed(n + steps)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    dy = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(*(() if lens is None else (len(lens),)), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    wt = (torch.randn(*(() if lens is None else (len(lens),)), k, 128, generator=g) * 0.05).bfloat16().to(gpu)
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    xq = K.quantize_mx_impl(x, afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
    wq = K.quantize_mx_weight_2d_impl(w, wfmt, rowwise=True, colwise=False, pad_to=128, kchunk=lay)
    run = lambda t: K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=lay, tile=t)
    assert torch.equal(run(tile).view(torch.int16), run("256").view(torch.int16))
    if afmt == wfmt and tile == "64x128":
        dq = K.quantize_mx_impl(dy, afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
        tq = K.quantize_mx_weight_2d_impl(wt, wfmt, rowwise=True, colwise=True, pad_to=128, kchunk=lay, col_scales_only=True)
        run = lambda t: K.grouped_gemm_mx_nt_impl(dq[0], dq[1], tq[0], tq[3], gl, kchunk=lay, b_transposed=True, tile=t)
        assert torch.equal(run(tile).view(torch.int16), run("256").view(torch.int16))
