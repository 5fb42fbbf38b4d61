"""The choice of an operand layout from sizes that are no plain integers: the symbols and tensors a tracer puts in their place."""

import numpy as np
import torch
from torch.fx.experimental.proxy_tensor import make_fx

from primus_amd.pytorch import kernels as K


def test_symbolic_sizes():
    seen = []

    def f(x, w):
        seen.append(type(x.shape[0]))
        return x * K.pick_layout(1, w.shape[0], w.shape[1], x.shape[0])

    traced = make_fx(f, tracing_mode="symbolic")(torch.ones(64, 128), torch.ones(96, 128))
    assert seen == [torch.SymInt]
    assert torch.equal(traced(torch.ones(64, 128), torch.ones(96, 128)), torch.full((64, 128), float(K.LAYOUT_KSTEP)))


def test_sizes_in_tensors_are_not_kept():
    before = K._kchunk_fits.cache_info().currsize
    for wrap in (torch.tensor, np.int64):
        assert K.kchunk_fits(wrap(3), wrap(3333), wrap(7777), wrap(999))
        assert not K.kchunk_fits(wrap(256), wrap(3333), wrap(7777), wrap(999))
    assert K._kchunk_fits.cache_info().currsize == before
    assert K.kchunk_fits(3, 3333, 7777, 999) and not K.kchunk_fits(256, 3333, 7777, 999)
    assert K._kchunk_fits.cache_info().currsize == before + 2
