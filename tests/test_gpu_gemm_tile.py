"""The small-tile GEMM kernel against the ring kernel on the same operands: every tile gives the same bits (each output
element runs the same MFMAs in the same order), on sizes that fill no tile, end inside a scale panel, and on ragged, short
and empty groups."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = ("64", "64x128", "128", None)
# k: 1, 2, 3, 5 and 9 K steps of 128 elements and one past a panel; rows around the tile heights
SHAPES = [(1, 32, 128), (63, 96, 160), (65, 160, 384), (129, 384, 640), (257, 128, 1152), (300, 544, 512)]
GROUPS = [([33, 0, 130, 1, 92, 300, 0, 257], 320, 384), ([0, 0, 64, 0], 128, 256), ([1] * 70 + [0, 129], 96, 128),
          ([(37 * i) % 97 if i % 5 else 0 for i in range(256)], 64, 128)]


def _same(x, y):
    return torch.equal(x.view(torch.uint8), y.view(torch.uint8))


def _operands(gpu, recipe, lens, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    dy = torch.randn(m, n, generator=g).bfloat16().to(gpu)
    w = (torch.randn(*(() if lens is None else (len(lens),)), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    return x, dy, w, gl


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4", "tensorwise"])
@pytest.mark.parametrize("lens,n,k", [(None, n, k) for _, n, k in SHAPES] + GROUPS)
def test_every_tile_gives_the_same_bits(gpu, recipe, lens, n, k):
    from primus_amd.pytorch import kernels as K

    m = dict((s[1:], s[0]) for s in SHAPES)[(n, k)] if lens is None else sum(lens)
    x, dy, w, gl = _operands(gpu, recipe, lens, m, n, k)
    aligned = n % 128 == 0 and k % 128 == 0
    if recipe == "tensorwise":
        xq = K.quantize_tensorwise_impl(x, 0, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
        dq = K.quantize_tensorwise_impl(dy, 2, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
        wq = K.quantize_weight_tensorwise_impl(w, 0, rowwise=True, colwise=True, pad_to=128, kchunk=2)
        runs = [lambda t: K.gemm_tw_nt_impl(xq[0], xq[1], xq[4], wq[0], wq[1], wq[4], gl, kchunk=2, tile=t),
                lambda t: K.gemm_tw_nt_impl(dq[0], dq[1], dq[4], wq[2], wq[3], wq[4], gl, kchunk=2, tile=t),
                lambda t: K.gemm_tw_wgrad_impl(dq[2], dq[3], dq[4], xq[2], xq[3], xq[4], gl, m, kchunk=2, tile=t)]
        if aligned:
            runs.append(lambda t: K.gemm_tw_nt_impl(dq[0], dq[1], dq[4], wq[0], wq[1], wq[4], gl, kchunk=2, b_transposed_n=k, tile=t))
    else:
        afmt, wfmt, lay = {"mxfp8": (0, 0, 2), "mxfp4w8": (0, 1, 2), "mxfp4": (1, 1, 3)}[recipe]
        xq = K.quantize_mx_impl(x, afmt, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        dq = K.quantize_mx_impl(dy, afmt, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        wq = K.quantize_mx_weight_2d_impl(w, wfmt, rowwise=True, colwise=True, pad_to=128, kchunk=lay)
        runs = [lambda t: K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=lay, tile=t),
                lambda t: K.grouped_gemm_mx_nt_impl(dq[0], dq[1], wq[2], wq[3], gl, kchunk=lay, tile=t)]
        if afmt == wfmt:
            runs.append(lambda t: K.grouped_gemm_mx_wgrad_impl(dq[2], dq[3], xq[2], xq[3], gl, m, kchunk=lay, tile=t))
            if aligned:
                runs.append(lambda t: K.grouped_gemm_mx_nt_impl(dq[0], dq[1], wq[0], wq[3], gl, kchunk=lay, b_transposed=True, tile=t))
    for i, run in enumerate(runs):
        want = run("256")
        for t in TILES:
            assert _same(run(t), want), (i, t)
