"""Activations and weight quantised in one launch (a linear's forward in one call) against a launch each: output, the bytes of
every copy, its scales and the tensor-wise factors, on plain, RMSNorm and Hadamard-transformed inputs; rows and columns that end
inside a tile, a scale panel and a supertile of the launch's tile order, one row, ragged and empty groups, weights with and
without a transposed copy of the codes."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4", "tensorwise"])
@pytest.mark.parametrize("lens,rows,n,k", [(None, 1, 32, 32), (None, 129, 160, 544), (None, 515, 640, 512), (None, 1100, 128, 4224),
                                           ([0, 130, 1, 0, 300, 64], 495, 256, 640), ([7, 0], 7, 96, 1056)])
def test_one_launch_writes_what_two_write(gpu, recipe, lens, rows, n, k):
    from primus_amd import _lib
    from primus_amd.pytorch import kernels as K

    tw = recipe == "tensorwise"
    fmt, lay = (_lib.FMT_E2M1, K.LAYOUT_KSTEP128) if recipe == "mxfp4" else (_lib.FMT_E4M3, K.LAYOUT_KSTEP)
    g = torch.Generator().manual_seed(rows + n + k)
    G = 0 if lens is None else len(lens)
    x = torch.randn(rows, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(*((G,) if G else ()), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    x[0, 0], w.view(-1)[-1] = float("inf"), 3e38
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    bt = n % 128 == 0 and k % 128 == 0
    # the call, on buffers filled beforehand
    plan = K.LinearPlan(rows=rows, n=n, k=k, groups=G, recipe=_lib.LINEAR_TENSORWISE if tw else _lib.LINEAR_MX, act_fmt=fmt, w_fmt=fmt,
                        grad_fmt=fmt, scale_mode=0, need_dx=1, need_dw=1, dx_from_rows=bt, w_quantized=0, input=_lib.LINEAR_PLAIN,
                        probs_dtype=0, grad_sr=0, rht_signs=-1, eps=0.0)
    saved = torch.full((plan.saved_bytes,), 0xA5, dtype=torch.uint8, device=gpu)
    scratch = torch.full((plan.fwd_bytes,), 0xA5, dtype=torch.uint8, device=gpu)
    y = torch.empty(rows, n, dtype=torch.bfloat16, device=gpu)
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.load().mxl_linear_forward(plan.ptr, x.data_ptr(), None, None, w.data_ptr(), None, ptr(gl), saved.data_ptr(), scratch.data_ptr(),
                                        y.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    # a launch each
    if tw:
        a = K.quantize_tensorwise_impl(x, fmt, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        b = K.quantize_weight_tensorwise_impl(w, fmt, rowwise=True, colwise=not bt, pad_to=128, kchunk=lay)
        want = K.gemm_tw_nt_impl(a[0], a[1], a[4], b[0], b[1], b[4], gl, kchunk=lay)
    else:
        a = K.quantize_mx_impl(x, fmt, rowwise=True, colwise=True, group_lens=gl, pad_to=128, kchunk=lay)
        b = K.quantize_mx_weight_2d_impl(w, fmt, rowwise=True, colwise=True, pad_to=128, kchunk=lay, col_scales_only=bt)
        if gl is None:
            want = K.gemm_mx_nt_impl(a[0], a[1], b[0], b[1], kchunk=lay)
        else:
            want = K.grouped_gemm_mx_nt_impl(a[0], a[1], b[0], b[1], gl, kchunk=lay)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    # every code array (they are written whole) is somewhere in the two buffers, at a multiple of 256 bytes
    hay = [bytes(t.cpu().numpy()) for t in (saved, scratch)]
    for codes in (a[0], a[2], b[0], b[2]):
        if codes is None or codes.numel() == 0:
            continue
        data = bytes(codes.contiguous().view(torch.uint8).cpu().numpy())
        assert any(h[i:i + len(data)] == data for h in hay for i in range(0, len(h) - len(data) + 1, 256))


# every byte of the two buffers, pieces that no launch writes (filled beforehand) among them
@pytest.mark.parametrize("kind", ["mxfp8", "mxfp4", "tensorwise", "mxfp8 norm", "mxfp4 signs"])
@pytest.mark.parametrize("lens,rows,n,k", [(None, 1, 32, 32), (None, 129, 160, 544), (None, 515, 640, 512), (None, 1100, 128, 4224),
                                           ([0, 130, 1, 0, 300, 64], 495, 256, 640), ([7, 0], 7, 96, 1056)])
def test_every_byte(gpu, kind, lens, rows, n, k):
    from primus_amd import _lib
    from primus_amd.pytorch import kernels as K

    if "norm" in kind and lens is not None:
        lens = None                       # the normalisation belongs to dense linears
    recipe, _, extra = kind.partition(" ")
    tw, fp4 = recipe == "tensorwise", recipe == "mxfp4"
    fmt = _lib.FMT_E2M1 if fp4 else _lib.FMT_E4M3
    g = torch.Generator().manual_seed(rows + n + k)
    G = 0 if lens is None else len(lens)
    x = torch.randn(rows, k, generator=g).bfloat16().to(gpu)
    w = (torch.randn(*((G,) if G else ()), n, k, generator=g) * 0.05).bfloat16().to(gpu)
    nw = torch.randn(k, generator=g).bfloat16().to(gpu)
    x[0, 0], w.view(-1)[-1] = float("inf"), 3e38
    gl = None if lens is None else torch.tensor(lens, dtype=torch.int64, device=gpu)
    bt = n % 128 == 0 and k % 128 == 0
    signs = 0xA6C9 if extra == "signs" else None
    plan = K.LinearPlan(rows=rows, n=n, k=k, groups=G, recipe=_lib.LINEAR_TENSORWISE if tw else _lib.LINEAR_MX, act_fmt=fmt, w_fmt=fmt,
                        grad_fmt=fmt, scale_mode=0, need_dx=1, need_dw=1, dx_from_rows=bt, w_quantized=0,
                        input=_lib.LINEAR_RMSNORM if extra == "norm" else _lib.LINEAR_PLAIN, probs_dtype=0, grad_sr=0,
                        rht_signs=-1 if signs is None else signs, eps=1e-5)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    fill = lambda b: torch.full((b,), 0xA5, dtype=torch.uint8, device=gpu)
    lens_ptr = None if gl is None else gl.data_ptr()
    saved, scratch = fill(plan.saved_bytes), fill(plan.fwd_bytes)
    y = torch.empty(rows, n, dtype=torch.bfloat16, device=gpu)
    assert lib.mxl_linear_forward(plan.ptr, x.data_ptr(), nw.data_ptr() if extra == "norm" else None, None, w.data_ptr(), None, lens_ptr,
                                  saved.data_ptr(), scratch.data_ptr(), y.data_ptr(), st) == 0
    # a launch each, into the same places of two other buffers
    saved2, scratch2 = fill(plan.saved_bytes), fill(plan.fwd_bytes)
    used = {id(saved2): 0, id(scratch2): 0}

    def take(buf, nbytes):
        at = used[id(buf)]
        used[id(buf)] = at + (nbytes + 255) // 256 * 256
        return buf.data_ptr() + at

    up = lambda v: (v + 127) // 128 * 128
    batch, per, W = G or 1, 2 if fp4 else 1, K.padded_width(rows, G)
    copy = lambda buf, r, ld, restarts=0: (take(buf, r * ld // per), take(buf, ((ld + 511) // 512 + restarts) * r * 16))
    x_col = copy(saved2, k, W, G + 1 if G else 0)
    w_row = copy(saved2, batch * n, up(k)) if bt else None
    w_col = (None, None)
    if not (tw and bt):
        w_col = (None if bt else take(saved2, batch * k * up(n) // per), take(saved2, (up(n) + 511) // 512 * batch * k * 16))
    rstd = take(saved2, rows * 4) if extra == "norm" else None
    x_si, w_si = (take(saved2, 4), take(saved2, 4)) if tw else (None, None)
    x_row = copy(scratch2, rows, up(k))
    w_row = w_row or copy(scratch2, batch * n, up(k))
    end = used[id(scratch2)]              # (behind it, tensor-wise: the workgroups' abs-max)
    qf = _lib.QF_KSTEP | (_lib.QF_KSTEP128 if fp4 else 0)
    if tw:
        ax, aw = torch.zeros(1, device=gpu), torch.zeros(1, device=gpu)
        assert lib.mxl_amax(x.data_ptr(), x.numel(), ax.data_ptr(), st) == 0 and lib.mxl_amax(w.data_ptr(), w.numel(), aw.data_ptr(), st) == 0
        assert lib.mxl_quantize_tensorwise(x.data_ptr(), rows, k, up(k), fmt, ax.data_ptr(), lens_ptr, G, *x_row, *x_col, x_si, qf, st) == 0
        assert lib.mxl_quantize_weight_tensorwise(w.data_ptr(), batch, n, k, up(k), up(n), fmt, aw.data_ptr(), *w_row, *w_col, w_si, qf, st) == 0
    else:
        if extra == "norm":
            assert lib.mxl_rmsnorm_fwd(x.data_ptr(), nw.data_ptr(), 1e-5, rows, k, None, rstd, st) == 0
            assert lib.mxl_rmsnorm_quantize(x.data_ptr(), nw.data_ptr(), rstd, rows, k, up(k), fmt, 0, None, 0, *x_row, *x_col, qf, st) == 0
        else:
            rht = _lib.QF_RHT_COL if signs is not None else 0
            assert lib.mxl_quantize_ex(x.data_ptr(), rows, k, up(k), fmt, 0, lens_ptr, G, *x_row, *x_col, qf | rht, 0, signs or 0, st) == 0
        assert lib.mxl_quantize_weight_2d_ex(w.data_ptr(), batch, n, k, up(k), up(n), fmt, 0, *w_row, *w_col, qf, st) == 0
    assert used[id(saved2)] == plan.saved_bytes and end == plan.fwd_bytes - (4096 if tw else 0)
    assert torch.equal(saved, saved2) and torch.equal(scratch[:end], scratch2[:end])
    last = (x_si, w_si, _lib.GF_KSTEP, st) if tw else (_lib.GF_KSTEP, st)
    want = torch.empty_like(y)
    gemm = lib.mxl_grouped_gemm_nt_scaled if tw else lib.mxl_grouped_gemm_nt_ex
    assert gemm(x_row[0], x_row[1], fmt, w_row[0], w_row[1], fmt, want.data_ptr(), lens_ptr, batch, rows, n, up(k), *last) == 0
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
