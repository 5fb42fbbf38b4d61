"""The row-wise copy alone of few rows (a wave on two rows of a scale panel) against the same copy out of the call that writes the
transposed one too, which works in 128 x 128 tiles: the same bytes at odd row counts, part-filled K steps and panels, for blocks
with infinities and NaN, every rounding of the scales, and inputs formed on the way."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("kind", ["plain", "norm", "silu", "gelu"])
@pytest.mark.parametrize("rows,cols", [(1, 32), (2, 96), (3, 512), (64, 544), (129, 1120), (255, 2880), (2047, 4096), (2049, 4096), (1536, 4096), (1537, 4096), (12288, 96), (12289, 96), (16384, 96), (16385, 96)])
def test_row_wise_copy_alone(gpu, fmt, kind, rows, cols):
    from primus_amd.pytorch import kernels as K

    g = torch.Generator().manual_seed(rows + cols)
    wide = cols * (2 if kind in ("silu", "gelu") else 1)
    x = (torch.randn(rows, wide, generator=g) * torch.logspace(-3, 3, wide)[torch.randperm(wide, generator=g)]).bfloat16()
    x[rows // 2, 5], x[rows - 1, cols - 1], x[0, cols // 2] = float("inf"), float("nan"), 3.0e38
    x[rows // 3, :32] = 0
    x = x.to(gpu)
    w = torch.randn(cols, generator=g).bfloat16().to(gpu)
    probs = torch.rand(rows, generator=g).to(gpu)
    mask = (torch.arange(rows) % 5 != 1).to(gpu)
    rstd = torch.rand(rows, generator=g).to(gpu) + 0.5

    def quantise(mode, colwise):
        if kind == "plain":
            return K.quantize_mx_impl(x, fmt, mode, rowwise=True, colwise=colwise, kchunk=K.LAYOUT_KSTEP)
        if kind == "norm":
            return K.rmsnorm_quantize_impl(x, w, rstd, fmt, mode, colwise=colwise, kchunk=K.LAYOUT_KSTEP)
        return K.glu_with_probs_quantize_impl(x, probs, mask, kind, fmt, mode, colwise=colwise, kchunk=K.LAYOUT_KSTEP)

    for mode in (0, 1, 2):
        got, want = quantise(mode, False), quantise(mode, True)
        assert torch.equal(got[0].view(torch.uint8), want[0].view(torch.uint8))
        s, t = got[1].view(torch.uint8), want[1].view(torch.uint8)
        # the last panel's bytes behind the padded row are written by neither
        last = (cols + 127) // 128 * 4 - (s.shape[0] - 1) * 16
        keep = torch.tensor([8 * (b & 1) + (b >> 1) for b in range(last)], device=gpu)
        assert torch.equal(s[:-1], t[:-1]) and torch.equal(s[-1][:, keep], t[-1][:, keep])
