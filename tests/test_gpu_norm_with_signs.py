"""``mxl_linear_forward`` on an input an RMSNorm forms: Hadamard signs, which belong to plain inputs, leave the forward as it is."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_the_forward_takes_no_notice_of_the_signs(gpu):
    from primus_amd import _lib
    from primus_amd.pytorch import kernels as K

    rows, n, k, fmt = 70, 128, 256, _lib.FMT_E2M1
    g = torch.Generator().manual_seed(1)
    x, w, nw = (torch.randn(*s, generator=g).bfloat16().to(gpu) for s in ((rows, k), (n, k), (k,)))
    y = [K.linear_forward_impl(K.linear_plan(rows, n, k, 0, _lib.LINEAR_MX, fmt, fmt, fmt, 0, True, True, True, False, _lib.LINEAR_RMSNORM,
                                             rht_signs=signs, eps=1e-5), x, w, aux0=nw)[0] for signs in (None, 0xA6C9)]
    assert torch.equal(*y)
