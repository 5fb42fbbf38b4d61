"""Stochastic rounding to E2M1 where a code changes: magnitudes at, just below and just above the point at which the element's own
random number carries them to the next code, below the smallest code where the point falls between integers, against the oracle."""

import numpy as np
import pytest
import torch

from oracle import mx_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [-100, 0, 90])
def test_magnitudes_around_their_crossing(gpu, scale):
    from primus_amd.pytorch import kernels as K

    rows, cols, seed = 512, 1024, (3 << 32) + 19
    words = o.sr_word(np.arange(rows * cols // 2, dtype=np.uint64), seed, 0)
    rnd = np.stack([words & np.uint32(0xFFFF), words >> np.uint32(16)], axis=-1).reshape(rows, cols).astype(np.int64)
    need = (1 << 22) - 64 * rnd                     # in units of 2^-23 (of 2^-22 from 1 on): this much and the code changes
    g = np.random.default_rng(7)
    delta = g.choice([-1.0, -0.5, -0.25, 0.0, 0.25, 0.5, 1.0], size=need.shape)
    low = np.clip(need + delta, 0, None) * 2.0 ** -23                        # below 0.5
    half = 0.5 + np.clip(need + delta, 0, (1 << 22) - 1) * 2.0 ** -23        # 0.5 to 1
    line = 1.0 + np.clip(need + delta, 0, (1 << 22) - 1) * 2.0 ** -23        # 1 to 1.5
    x = np.choose(g.integers(0, 3, size=need.shape), [low, half, line]) * g.choice([-1.0, 1.0], size=need.shape)
    x[:, ::32] = 4.0                                # the block's maximum: w = x
    x = (torch.from_numpy(x) * 2.0 ** scale).bfloat16()
    q, s, _, _ = K.quantize_mx_impl(x.to(gpu), o.FMT_E2M1, rowwise=True, sr_seed=seed)
    want, want_s = o.quantize_mx_rowwise_sr(x, seed)
    assert np.array_equal(s.view(torch.uint8).cpu().numpy(), want_s)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), want)
