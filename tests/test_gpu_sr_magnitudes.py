"""Stochastic rounding to E2M1 over every bf16 magnitude a block can hold: the branch-free magnitude against the oracle,
from far below the smallest code to the saturated one, both signs, in both copies, with bit-equal codes."""

import numpy as np
import pytest
import torch

from oracle import mx_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [0, -100, 90])      # of the block maximum: scale bytes in the middle and near both ends
@pytest.mark.parametrize("seed", [0, (5 << 32) + 77])
def test_every_magnitude_below_the_block_maximum(gpu, exponent, seed):
    from primus_amd.pytorch import kernels as K

    # 128 mantissas of 20 octaves and zero, in both signs, dealt to blocks whose first element fixes the scale
    m = (1.0 + torch.arange(128) / 128.0).double()
    v = torch.cat([m * 2.0 ** e for e in range(-18, 2)] + [torch.zeros(1).double()]) * 2.0 ** exponent
    v = torch.cat([v, -v])
    g = torch.Generator().manual_seed(11)
    x = v[torch.randint(0, v.numel(), (160, 256), generator=g)]
    x[:, ::32] = 3.984375 * 2.0 ** exponent
    x[::32, :] = -3.984375 * 2.0 ** exponent
    x = x.bfloat16()
    q, s, qt, st = K.quantize_mx_impl(x.to(gpu), o.FMT_E2M1, rowwise=True, colwise=True, sr_seed=seed)
    want, want_s = o.quantize_mx_rowwise_sr(x, seed)
    want_t, want_st = o.quantize_mx_colwise_segmented_sr(x, [160], seed)
    for got, ref in ((q, want), (s, want_s), (qt, want_t), (st, want_st)):
        assert np.array_equal(got.view(torch.uint8).cpu().numpy(), ref)
