"""The scan over group_lens that every grouped kernel starts with, where it can go wrong: group counts around and past the 64
that a wave sums up at once, empty groups across those seams, and counts that do not match the buffer (negative, or more rows
than there are)."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _lens(G, kind):
    if kind == "edges":        # rows only around the seams of 64
        return [(7 * i) % 150 if i % 64 in (0, 1, 62, 63) or i == G - 1 else 0 for i in range(G)]
    return [1 + (5 * i) % 9 for i in range(G)]


@pytest.mark.parametrize("kind", ["edges", "all"])
@pytest.mark.parametrize("G", [2, 63, 64, 65, 129, 256])
def test_every_group_gets_its_own_rows(gpu, G, kind):
    from primus_amd.pytorch import kernels as K

    lens, n, k = _lens(G, kind), 64, 128
    m = sum(lens)
    gen = torch.Generator().manual_seed(G)
    # entries of a few bits: every product and sum is exact, whatever the order
    x, dy = (torch.randint(-2, 3, (m, c), generator=gen).bfloat16().to(gpu) for c in (k, n))
    w = torch.randint(-2, 3, (G, n, k), generator=gen).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    xq = K.quantize_mx_impl(x, 0, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
    dq = K.quantize_mx_impl(dy, 0, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
    wq = K.quantize_mx_weight_2d_impl(w, 0, rowwise=True, colwise=False, pad_to=128, kchunk=2)
    off = np.cumsum([0] + lens)
    want_y = torch.cat([x[off[i]:off[i + 1]].float() @ w[i].float().t() for i in range(G)]).bfloat16()
    want_dw = torch.stack([dy[off[i]:off[i + 1]].float().t() @ x[off[i]:off[i + 1]].float() for i in range(G)]).bfloat16()
    for tile in ("256", "128", "64x128"):
        assert torch.equal(K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=2, tile=tile), want_y), tile
        assert torch.equal(K.grouped_gemm_mx_wgrad_impl(dq[2], dq[3], xq[2], xq[3], gl, m, kchunk=2, tile=tile), want_dw), tile
    assert torch.equal(K.grouped_gemm_bf16_impl(x, w, gl), want_y)
    assert torch.equal(K.grouped_gemm_bf16_wgrad_impl(dy, x, gl), want_dw)
    # row-major operands: the two-slot kernel
    rq = K.quantize_mx_impl(x, 0, rowwise=True, colwise=False, pad_to=128)
    vq = K.quantize_mx_weight_2d_impl(w, 0, rowwise=True, colwise=False, pad_to=128)
    assert torch.equal(K.grouped_gemm_mx_nt_impl(rq[0], rq[1], vq[0], vq[1], gl), want_y)


@pytest.mark.parametrize("G", [3, 64, 70])
def test_counts_that_do_not_match_the_buffer(gpu, G):
    """Negative counts read as 0 and the running sum never passes the rows there are: the same copies as with the counts that
    this comes to."""
    from primus_amd.pytorch import kernels as K

    rows, cols = 300, 64
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(G)).bfloat16().to(gpu)
    bad = [-5, 170, 1 << 40] + [3] * (G - 3)
    good = [0, 170, 130] + [0] * (G - 3)
    a, b = (K.quantize_mx_impl(x, 0, rowwise=True, colwise=True, group_lens=torch.tensor(v, dtype=torch.int64, device=gpu), pad_to=128,
                               kchunk=2) for v in (bad, good))
    assert torch.equal(a[0].view(torch.uint8), b[0].view(torch.uint8))
    assert torch.equal(a[2].view(torch.uint8)[: 2 * 4], b[2].view(torch.uint8)[: 2 * 4])      # (the steps of the two groups that have rows)


@pytest.mark.parametrize("G", [3, 64, 70])
def test_the_gemms_clamp_the_counts_too(gpu, G):
    """The same in every kernel that multiplies by group: rows in the forward; in the weight gradient negative counts, and a last group
    whose count passes the padded width (each segment one row past a whole one, so that the segments fill that width)."""
    from primus_amd.pytorch import kernels as K

    n, k = 64, 128
    gen = torch.Generator().manual_seed(G)

    def counts(v):
        return torch.tensor(v, dtype=torch.int64, device=gpu)

    def ints(*shape):      # every product and sum is exact
        return torch.randint(-2, 3, shape, generator=gen).bfloat16().to(gpu)

    def by_hand(dy, x, lens):
        off = np.cumsum([0] + lens)
        return torch.stack([dy[off[i]:off[i + 1]].float().t() @ x[off[i]:off[i + 1]].float() for i in range(G)]).bfloat16()

    lens, bad = [0, 170, 130] + [0] * (G - 3), counts([-5, 170, 1 << 40] + [3] * (G - 3))
    x, dy, w = ints(300, k), ints(300, n), ints(G, n, k)
    want = torch.cat([x[:170].float() @ w[1].float().t(), x[170:].float() @ w[2].float().t()]).bfloat16()
    for layout in (0, 1, 2):
        a, b = (f(t, 0, rowwise=True, colwise=False, pad_to=128, kchunk=layout) for f, t in ((K.quantize_mx_impl, x), (K.quantize_mx_weight_2d_impl, w)))
        for tile in ("256", "128", "64x128", "64") if layout == 2 else (None,):
            assert torch.equal(K.grouped_gemm_mx_nt_impl(a[0], a[1], b[0], b[1], bad, kchunk=layout, tile=tile), want), (layout, tile)
    for tile in (128, 256):
        assert torch.equal(K.grouped_gemm_bf16_impl(x, w, bad, tile=tile), want), tile
        assert torch.equal(K.grouped_gemm_bf16_wgrad_impl(dy, x, bad, tile=tile), by_hand(dy, x, lens)), tile

    full = [129] + [1] * (G - 1)
    for lens, bad in (([0, 170, 130] + [0] * (G - 3), [-5, 170, 130] + [-1 << 40] * (G - 3)), (full, full[:-1] + [1 << 40])):
        m = sum(lens)
        want = by_hand(dy[:m], x[:m], lens)
        for layout in (0, 1, 2):
            p, q = (K.quantize_mx_impl(t[:m], 0, rowwise=False, colwise=True, group_lens=counts(lens), pad_to=128, kchunk=layout) for t in (dy, x))
            for tile in ("256", "128", "64x128", "64") if layout == 2 else (None,):
                got = K.grouped_gemm_mx_wgrad_impl(p[2], p[3], q[2], q[3], counts(bad), m, kchunk=layout, tile=tile)
                assert torch.equal(got, want), (layout, tile)
