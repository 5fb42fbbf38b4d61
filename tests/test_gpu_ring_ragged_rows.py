"""The ring kernel's tiles at a group's ragged end: row counts on both sides of every number of live fragments (64, 128, 192,
256 rows), alone and behind a whole tile, and column counts on both sides of the output patches (64 and 128 columns).  Compared
bit for bit with the 128 x 128 tile, which runs the same MFMAs per output element; rows and columns next to the tile must stay
untouched, so the output is one part of a larger buffer filled beforehand.  The last sizes of each list give a workgroup
several tiles, one behind the other's stores."""

import ctypes

import pytest
import torch

from primus_amd import _lib

pytestmark = pytest.mark.gpu

LENS = [1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 384, 448, 449]
GUARD = 512


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4"])
@pytest.mark.parametrize("n,k", [(32, 128), (64, 256), (96, 384), (160, 128), (320, 640), (512, 128), (4096, 128)])
def test_ragged_tiles(gpu, recipe, n, k):
    from primus_amd.pytorch import kernels as K

    afmt, wfmt, lay = {"mxfp8": (0, 0, 2), "mxfp4w8": (0, 1, 2), "mxfp4": (1, 1, 3)}[recipe]
    g = torch.Generator().manual_seed(n + k)
    m, G = sum(LENS), len(LENS)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(G, n, k, generator=g) * 0.05).bfloat16().to(gpu)
    gl = torch.tensor(LENS, dtype=torch.int64, device=gpu)
    xq = K.quantize_mx_impl(x, afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
    wq = K.quantize_mx_weight_2d_impl(w, wfmt, rowwise=True, colwise=False, pad_to=128, kchunk=lay)
    want = K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=lay, tile="128")
    buf = torch.full((GUARD + m * n + GUARD,), 7.0, dtype=torch.bfloat16, device=gpu)
    out = buf[GUARD:GUARD + m * n]
    p = ctypes.c_void_p
    rc = _lib.load().mxl_grouped_gemm_nt_ex(p(xq[0].data_ptr()), p(xq[1].data_ptr()), afmt, p(wq[0].data_ptr()), p(wq[1].data_ptr()), wfmt,
                                            p(out.data_ptr()), p(gl.data_ptr()), G, m, n, k, _lib.GF_KSTEP | _lib.GF_TILES["256"],
                                            p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert torch.equal(out.view(m, n).view(torch.int16), want.view(torch.int16))
    assert bool((buf[:GUARD] == 7.0).all()) and bool((buf[GUARD + m * n:] == 7.0).all())


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4"])
@pytest.mark.parametrize("n,k", [(32, 64), (96, 320), (288, 160), (416, 480), (2080, 2048)])
def test_weight_gradient_edges(gpu, recipe, n, k):
    from primus_amd.pytorch import kernels as K

    fmt, lay = {"mxfp8": (0, 2), "mxfp4": (1, 3)}[recipe]
    lens = [130, 0, 513, 64, 128, 1]
    g = torch.Generator().manual_seed(n * k)
    m, G = sum(lens), len(lens)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    dy = torch.randn(m, n, generator=g).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    xq = K.quantize_mx_impl(x, fmt, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
    dq = K.quantize_mx_impl(dy, fmt, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
    want = K.grouped_gemm_mx_wgrad_impl(dq[2], dq[3], xq[2], xq[3], gl, m, kchunk=lay, tile="128")
    got = K.grouped_gemm_mx_wgrad_impl(dq[2], dq[3], xq[2], xq[3], gl, m, kchunk=lay, tile="256")
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# 11 x 24 tiles on 256 workgroups (a last round of 8, run as 16 halves): a last row tile with rows in both halves, in one
# (exactly full, and not), and a ragged last column tile; and fewer tiles than half of the workgroups a grouped launch has
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4w8", "mxfp4"])
@pytest.mark.parametrize("lens,n", [((2700,), 6112), ((2688,), 6144), ((2590,), 6112), ((2800, 16), 5984), ((0, 3, 0, 0, 300, 0, 1, 0), 480)])
def test_last_round_in_halves(gpu, recipe, lens, n):
    from primus_amd.pytorch import kernels as K

    afmt, wfmt, lay = {"mxfp8": (0, 0, 2), "mxfp4w8": (0, 1, 2), "mxfp4": (1, 1, 3)}[recipe]
    m, k, G = sum(lens), 128, len(lens)
    g = torch.Generator().manual_seed(n + m)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(G, n, k, generator=g) * 0.05).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    xq = K.quantize_mx_impl(x, afmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
    wq = K.quantize_mx_weight_2d_impl(w, wfmt, rowwise=True, colwise=False, pad_to=128, kchunk=lay)
    got, want = (K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], gl, kchunk=lay, tile=t) for t in ("256", "128"))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "tensorwise"])
@pytest.mark.parametrize("m,n,k,grouped", [(70, 2720, 6112, False), (300, 2592, 6144, False), (640, 2688, 6112, False), (300, 2720, 6112, True)])
def test_weight_gradient_in_halves(gpu, recipe, m, n, k, grouped):
    from primus_amd.pytorch import kernels as K

    g = torch.Generator().manual_seed(n + m)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    dy = torch.randn(m, n, generator=g).bfloat16().to(gpu)
    gl = torch.tensor([m], dtype=torch.int64, device=gpu) if grouped else None      # (a single group: the tile order of groups)
    if recipe == "tensorwise":
        xq = K.quantize_tensorwise_impl(x, 0, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
        dq = K.quantize_tensorwise_impl(dy, 2, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=2)
        run = lambda t, into=None: K.gemm_tw_wgrad_impl(dq[2], dq[3], dq[4], xq[2], xq[3], xq[4], gl, m, kchunk=2, tile=t, accum_into=into)
    else:
        fmt, lay = {"mxfp8": (0, 2), "mxfp4": (1, 3)}[recipe]
        xq = K.quantize_mx_impl(x, fmt, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        dq = K.quantize_mx_impl(dy, fmt, rowwise=False, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        run = lambda t, into=None: K.grouped_gemm_mx_wgrad_impl(dq[2], dq[3], xq[2], xq[3], gl, m, kchunk=lay, tile=t, accum_into=into)
    got, want = run("256"), run("128")
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # added to a float32 buffer of zeros: the same sums before their rounding to bf16
    into = torch.zeros(want.shape, dtype=torch.float32, device=gpu)
    run(None, into)
    assert torch.equal(into.bfloat16().view(torch.int16), want.view(torch.int16))


# the same splits on transposed weight codes (every input gradient) and under per-tensor factors
@pytest.mark.parametrize("kind", ["mxfp8 transposed", "mxfp4 transposed", "e4m3 scaled", "e5m2 scaled", "e4m3 scaled transposed", "e5m2 scaled transposed"])
@pytest.mark.parametrize("lens,n", [((2700,), 6112), ((2688,), 6144), ((2590,), 6112), ((2800, 16), 5984), ((0, 3, 0, 0, 300, 0, 1, 0), 480)])
def test_last_round_in_halves_other_kernels(gpu, kind, lens, n):
    from primus_amd.pytorch import kernels as K

    m, k, G, bt = sum(lens), 128, len(lens), "transposed" in kind
    g = torch.Generator().manual_seed(n + m)
    x = torch.randn(m, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(G, *((k, n) if bt else (n, k)), generator=g) * 0.05).bfloat16().to(gpu)
    gl = torch.tensor(lens, dtype=torch.int64, device=gpu)
    if "scaled" in kind:
        xq = K.quantize_tensorwise_impl(x, _lib.FMT_E5M2 if "e5m2" in kind else _lib.FMT_E4M3, rowwise=True, colwise=False, pad_to=128, kchunk=2)
        wq = K.quantize_weight_tensorwise_impl(w, _lib.FMT_E4M3, rowwise=True, colwise=False, pad_to=128, kchunk=2)
        run = lambda t: K.gemm_tw_nt_impl(xq[0], xq[1], xq[4], wq[0], wq[1], wq[4], gl, kchunk=2, b_transposed_n=n if bt else None, tile=t)
    else:
        fmt, lay = {"mxfp8": (0, 2), "mxfp4": (1, 3)}[kind.split()[0]]
        xq = K.quantize_mx_impl(x, fmt, rowwise=True, colwise=False, group_lens=gl, pad_to=128, kchunk=lay)
        wq = K.quantize_mx_weight_2d_impl(w, fmt, rowwise=True, colwise=True, pad_to=128, kchunk=lay, col_scales_only=True)
        run = lambda t: K.grouped_gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[3], gl, kchunk=lay, b_transposed=True, tile=t)
    got, want = run("256"), run("128")
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# an output aligned to less than the stores' 16 bytes, inside a larger buffer
@pytest.mark.parametrize("offset", [0, 1, 2, 4])
@pytest.mark.parametrize("m,n", [(300, 96), (33, 320)])
def test_output_alignment(gpu, offset, m, n):
    from primus_amd.pytorch import kernels as K

    k = 256
    g = torch.Generator().manual_seed(n)
    xq = K.quantize_mx_impl(torch.randn(m, k, generator=g).bfloat16().to(gpu), 0, rowwise=True, colwise=False, pad_to=128, kchunk=2)
    wq = K.quantize_mx_weight_2d_impl(torch.randn(n, k, generator=g).bfloat16().to(gpu), 0, rowwise=True, colwise=False, pad_to=128, kchunk=2)
    want = K.gemm_mx_nt_impl(xq[0], xq[1], wq[0], wq[1], kchunk=2)
    buf = torch.full((GUARD + m * n + GUARD,), 7.0, dtype=torch.bfloat16, device=gpu)
    at = GUARD // 2 + offset
    rc = _lib.load().mxl_grouped_gemm_nt_ex(xq[0].data_ptr(), xq[1].data_ptr(), 0, wq[0].data_ptr(), wq[1].data_ptr(), 0, buf[at:].data_ptr(),
                                            None, 1, m, n, k, _lib.GF_KSTEP | _lib.GF_TILES["256"], torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(buf[at:at + m * n].view(m, n).view(torch.int16), want.view(torch.int16))
    assert bool((buf[:at] == 7.0).all()) and bool((buf[at + m * n:] == 7.0).all())
