"""The 256-row bf16 tiles where a slot of 64 contraction elements is not full: contractions of an odd number of halves
(forward, dgrad), groups of every remainder of tokens (wgrad), row tiles that leave whole waves or parts of them without
rows, column tiles that leave waves without columns, and workgroups that go on to further tiles while the first one's
output leaves.  Integer operands: every partial sum is exact, so the result equals the float32 matmul bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,n,k", [
    ([1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 161], 96, 32),
    ([256, 0, 257, 160, 1, 97], 320, 96),
    ([191, 193, 0, 0, 449], 32, 160),
    ([64 + i % 3 for i in range(200)], 544, 224),
    ([4096, 3840, 1], 4096, 64),
])
def test_exact_on_integers(gpu, lens, n, k):
    from primus_amd.pytorch import kernels as K

    G, m = len(lens), sum(lens)
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randint(-3, 4, (m, k), generator=gen).bfloat16().to(gpu)
    b = torch.randint(-2, 3, (G, n, k), generator=gen).bfloat16().to(gpu)
    dy = torch.randint(-2, 3, (m, n), generator=gen).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    y = K.grouped_gemm_bf16_impl(a, b, gl, tile=256)
    dx = K.grouped_gemm_bf16_impl(dy, b, gl, b_kn=True, tile=256)
    dw = K.grouped_gemm_bf16_wgrad_impl(dy, a, gl, tile=256)
    acc = torch.ones(G, n, k, dtype=torch.float32, device=gpu)
    K.grouped_gemm_bf16_wgrad_impl(dy, a, gl, accum_into=acc, tile=256)
    off = 0
    for g, ln in enumerate(lens):
        rows = slice(off, off + ln)
        assert torch.equal(y[rows], (a[rows].float() @ b[g].float().t()).bfloat16()), g
        assert torch.equal(dx[rows], (dy[rows].float() @ b[g].float()).bfloat16()), g
        want = dy[rows].float().t() @ a[rows].float()
        assert torch.equal(dw[g], want.bfloat16()), g
        assert torch.equal(acc[g], want + 1.0), g
        off += ln
