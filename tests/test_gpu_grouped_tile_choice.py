"""Grouped forward and dgrad on either side of the lines by which a launch picks its output tile: the tile it picks gives the bits of
the ring kernel (each output element runs the same MFMAs in the same order)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _lens(groups, rows):
    """Uneven, some empty, ``rows`` per group on average."""
    lens = [(2 * rows * (i % 5)) // 4 for i in range(groups)]
    lens[-1] += groups * rows - sum(lens)
    return lens


# more than 300 ring tiles each; k 256: weights of 192 MiB and less, k 3328: more (E2M1 weights count half)
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "mxfp4w8"])
@pytest.mark.parametrize("k,rows", [(256, 32), (256, 33), (256, 97), (256, 192), (256, 193), (3328, 16), (3328, 17), (3328, 32), (3328, 33), (3328, 65)])
def test_the_tile_a_grouped_launch_picks(gpu, recipe, k, rows):
    from primus_amd.pytorch import kernels as K

    groups, n = 64, 2560
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
