"""``mxl_linear_forward`` on an input an RMSNorm forms: a live row count (``lens`` next to ``groups`` = 0) reaches the GEMM alone."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live", [1, 50, 70])
def test_rows_up_to_the_count(gpu, live):
    from primus_amd import _lib
    from primus_amd.pytorch import kernels as K

    rows, n, k, fmt = 70, 128, 256, _lib.FMT_E4M3
    g = torch.Generator().manual_seed(1)
    x, w, nw = (torch.randn(*s, generator=g).bfloat16().to(gpu) for s in ((rows, k), (n, k), (k,)))
    plan = K.linear_plan(rows, n, k, 0, _lib.LINEAR_MX, fmt, fmt, fmt, 0, True, True, True, False, _lib.LINEAR_RMSNORM, eps=1e-5)
    want, saved = K.linear_forward_impl(plan, x, w, aux0=nw)
    got, saved_got = K.linear_forward_impl(plan, x, w, None, torch.tensor([live], device=gpu), nw)
    codes = k * 128                       # the transposed copy of the input comes first: 70 rows padded to 128
    assert torch.equal(got[:live], want[:live]) and torch.equal(saved_got[:codes], saved[:codes])
