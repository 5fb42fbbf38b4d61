"""Activations and weight quantised in one launch (a linear's forward in one call) against a launch each, on the bytes of every
copy: rows and columns that end inside a tile, a scale panel and a supertile of the launch's tile order, one row, ragged and
empty groups, weights with and without a transposed copy of the codes."""

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
