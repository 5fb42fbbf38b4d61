// One linear as two calls: everything its forward launches, and everything its backward launches (host code only).
//
// A linear is 2 to 4 launches forward and 2 to 5 backward, and a dozen buffers.  Issued one by one from Python, with an
// allocation per buffer and a stream look-up per launch, they take 230 us for a pass whose kernels need 60.  Here the
// caller allocates three buffers -- what the backward needs, and a scratch buffer per direction -- and makes one call per
// direction; the layout of the buffers is arithmetic on the sizes and is worked out again in every call.
#include "mx_activation.h"
#include "mx_gemm_tile.h"
#include "mx_quantize.h"
#include "mx_blockwise.h"

namespace {

int64_t rup(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// hands out pieces of a buffer; with base null it only counts
struct Arena {
    uint8_t* base;
    int64_t used = 0;
    explicit Arena(void* b) : base((uint8_t*)b) {}
    uint8_t* take(int64_t bytes) {
        uint8_t* p = base ? base + used : nullptr;
        used += rup(bytes, 256);
        return p;
    }
};

struct Copy {          // one quantised copy: codes, scales
    uint8_t *q = nullptr, *s = nullptr;
};

struct Linear {
    const mxl_linear& p;
    int64_t batch, k_ld, n_ld, width;
    int f44;
    explicit Linear(const mxl_linear* d) : p(*d) {
        batch = p.groups > 0 ? p.groups : 1;
        k_ld = rup(p.k, 128);
        n_ld = rup(p.n, 128);
        width = mxl_padded_width(p.rows, (int)p.groups);
        f44 = p.act_fmt == MXL_FMT_E2M1 && p.w_fmt == MXL_FMT_E2M1;
    }
    bool mx() const { return p.recipe == MXL_LINEAR_MX; }
    bool tensorwise() const { return p.recipe == MXL_LINEAR_TENSORWISE; }
    bool blockwise() const { return p.recipe == MXL_LINEAR_BLOCKWISE; }
    // Whether codes go through the caches (as far as they fit, mx_quantize.hip) or are streamed past them.  The GEMM behind reads
    // them next; what it does not find in the cache any more was written to memory while it multiplied instead of before.  So:
    // everything where a linear's operands fit the 256 MiB memory-side cache together, and beyond that where the GEMMs multiply
    // rather than read weights.  Not with tensor-wise scaling, whose quantiser finds its input in that cache, left there by the
    // abs-max pass.  us a pass, streamed / row-wise copies kept / both copies kept: [1999, 2880] x 5760 143 / 134 / 132, [8192, 4096] x
    // 4096 386 / 380 / 377, [4096, 4096] x 14336 639 / 631 / 623, [16384, 4096] x 14336 2296 / 2274 / 2283; E2M1 [8192, 8192] x 8192 828 /
    // 817 / 815; 16 experts of 1408, 2048 wide, 256 and 1024 rows each, 372 / 354 / 347 and 785 / 762 / 763; E2M1 weights, 128 experts
    // [5760, 2880], 512 rows each, 3996 / 3969 / 3970.  Bound by their weights: 32 experts [4096, 7168] and [7168, 2048], 256 rows each,
    // 2690 / 2740 / 2745 (forward GEMM 319 -> 352).  Tensor-wise, [4096, 4096] x 8192, 383 / 385 / 383.
    bool keeps() const {
        const int64_t copies = p.rows * (k_ld + n_ld) * 2 / (p.act_fmt == MXL_FMT_E2M1 ? 2 : 1) + batch * n_ld * k_ld / (p.w_fmt == MXL_FMT_E2M1 ? 2 : 1);
        return mx() && (p.rows >= 512 * batch || copies <= (int64_t)256 << 20);
    }
    uint32_t qf() const { return MXL_QF_KSTEP | (f44 ? MXL_QF_KSTEP128 : 0u); }

    // K-step-major copies of [rows, ld] (ld padded): codes, scale panels
    static Copy rows_copy(Arena& a, int64_t rows, int64_t ld, int64_t fmt, int64_t restarts = 0) {
        Copy c;
        c.q = a.take(rows * ld / (fmt == MXL_FMT_E2M1 ? 2 : 1));
        c.s = a.take(((ld + 511) / 512 + restarts) * rows * 16);
        return c;
    }
    Copy x_row(Arena& a) const { return rows_copy(a, p.rows, k_ld, p.act_fmt); }
    Copy cols_copy(Arena& a, int64_t cols, int64_t fmt) const { return rows_copy(a, cols, width, fmt, p.groups > 0 ? p.groups + 1 : 0); }
    // Rows per matrix of the weight's row-wise copy: where the backward reads it transposed, its rows are a contraction and each
    // matrix is filled up with zeros to whole K steps, which the forward steps over (a neighbouring expert's rows in their
    // place would meet zero codes of dy, but NaN among them would stay NaN).  With a transposed copy of the codes instead, for
    // widths that are no multiples of 128, the quantiser writes a byte more per element; a pass before and now, us: 32 experts of
    // [4544, 1152] and [1152, 2272], 284 rows, 480 -> 422; of [2176, 6816] and [6816, 1088], 8460 rows, 1871 -> 1733; E2M1, of
    // [4736, 2624] and [2624, 2368], 200 rows, 829 -> 770; dense, [1999, 2880] x 5760, 151 -> 143, E2M1 [2736, 8064] x 13408, 592 -> 578.
    int64_t w_rows() const { return p.need_dx && p.dx_from_rows ? n_ld : p.n; }
    Copy w_row(Arena& a) const { return rows_copy(a, batch * w_rows(), k_ld, p.w_fmt); }
    Copy w_col(Arena& a) const {
        Copy c;
        if (!p.dx_from_rows) c.q = a.take(batch * p.k * n_ld / (p.w_fmt == MXL_FMT_E2M1 ? 2 : 1));
        c.s = a.take((n_ld + 511) / 512 * batch * p.k * 16);
        return c;
    }
};

// what the forward leaves for the backward
struct Saved {
    Copy x_col, w_row, w_col;
    float *rstd = nullptr, *x_si = nullptr, *w_si = nullptr;
    Saved(const Linear& l, Arena& a) {
        const mxl_linear& p = l.p;
        if (p.need_dw) x_col = l.cols_copy(a, p.k, p.act_fmt);
        if (p.need_dx && !p.w_quantized) {
            if (p.dx_from_rows) w_row = l.w_row(a);
            if (!(l.tensorwise() && p.dx_from_rows)) w_col = l.w_col(a);
        }
        if (p.input == MXL_LINEAR_RMSNORM) rstd = (float*)a.take(p.rows * 4);
        if (l.tensorwise()) {
            x_si = (float*)a.take(4);
            w_si = (float*)a.take(4);
        }
    }
};
struct ForwardScratch {
    Copy x_row, w_row;
    float *x_amax = nullptr, *w_amax = nullptr;
    ForwardScratch(const Linear& l, Arena& a) {
        x_row = l.x_row(a);
        if (!l.p.w_quantized && !(l.p.need_dx && l.p.dx_from_rows)) w_row = l.w_row(a);
        if (l.tensorwise()) {
            x_amax = (float*)a.take(4 * mxl::AMAX_PARTS);
            w_amax = (float*)a.take(4 * mxl::AMAX_PARTS);
        }
    }
};
struct BackwardScratch {
    Copy d_row, d_col;
    float *amax = nullptr, *d_si = nullptr, *norm_ws = nullptr;
    int64_t norm_bytes = 0;
    void* dxi = nullptr;          // gradient of the GEMM's input where the operator's input is something else
    BackwardScratch(const Linear& l, Arena& a) {
        const mxl_linear& p = l.p;
        if (p.need_dx) d_row = Linear::rows_copy(a, p.rows, l.n_ld, p.grad_fmt);
        if (p.need_dw) d_col = l.cols_copy(a, p.n, p.grad_fmt);
        if (l.tensorwise()) {
            amax = (float*)a.take(4 * mxl::AMAX_PARTS);
            d_si = (float*)a.take(4);
        }
        if (p.input != MXL_LINEAR_PLAIN && p.need_dx) dxi = a.take(p.rows * p.k * 2);
        if (p.input == MXL_LINEAR_RMSNORM && p.need_dx) {
            norm_bytes = mxl_rmsnorm_bwd_workspace_bytes(p.rows, p.k);
            norm_bytes = norm_bytes < 16 ? 16 : norm_bytes;
            norm_ws = (float*)a.take(norm_bytes);
        }
    }
};

// The 128-blockwise recipe (forward and backward of [1024, 2048] x 2048 190 -> 108 us in two calls, [256, 4096] x 4096 191 ->
// 119; launch by launch it is bound by the host there).  Forward: row-wise copies of x and w.  Backward, from the bf16
// tensors: both copies of dy, the transposed ones of x and w.
struct BwForward {
    Copy x, w;
    BwForward(const Linear& l, Arena& a) {
        const mxl_linear& p = l.p;
        x.q = a.take(p.rows * p.k);
        x.s = a.take(p.rows * (p.k / 128) * 4);
        w.q = a.take(l.batch * p.n * p.k);
        w.s = a.take(l.batch * (p.n / 128) * (p.k / 128) * 4);
    }
};
struct BwBackward {
    Copy d_row, d_col, x_col, w_col;
    BwBackward(const Linear& l, Arena& a) {
        const mxl_linear& p = l.p;
        if (p.need_dx) {
            d_row.q = a.take(p.rows * p.n);
            d_row.s = a.take(p.rows * (p.n / 128) * 4);
            w_col.q = a.take(l.batch * p.k * p.n);
            w_col.s = a.take(l.batch * (p.k / 128) * (p.n / 128) * 4);
        }
        if (p.need_dw) {
            d_col.q = a.take(p.n * l.width);
            d_col.s = a.take(p.n * (l.width / 128) * 4);
            x_col.q = a.take(p.k * l.width);
            x_col.s = a.take(p.k * (l.width / 128) * 4);
        }
    }
};

bool valid(const mxl_linear* p) {
    if (!p || p->rows <= 0 || p->n <= 0 || p->k <= 0 || p->n % MXL_BLOCK || p->k % MXL_BLOCK || p->groups < 0 || p->groups > MXL_MAX_GROUPS) return false;
    if (p->recipe == MXL_LINEAR_BLOCKWISE) return p->input == MXL_LINEAR_PLAIN && !p->w_quantized && p->n % 128 == 0 && p->k % 128 == 0;
    if (p->recipe != MXL_LINEAR_MX && p->recipe != MXL_LINEAR_TENSORWISE) return false;
    if (p->recipe == MXL_LINEAR_TENSORWISE && (p->input != MXL_LINEAR_PLAIN || p->w_quantized)) return false;
    if (p->input < MXL_LINEAR_PLAIN || p->input > MXL_LINEAR_RMSNORM) return false;
    return !(p->dx_from_rows && p->w_quantized);
}

}  // namespace

#define MXL_TRY(call)                    \
    do {                                 \
        const int rc_ = (call);          \
        if (rc_ != MXL_OK) return rc_;   \
    } while (0)

namespace {

// As keeps() above, per launch of the quantiser: its codes fit the memory-side cache, or the GEMM multiplies rather than reads weights.
// us a pass, streamed / kept: [128, 4096] x 8192 179 / 146, [1024, 4096] x 4096 132 / 120, [3000, 7168] x 2048 228 / 209, [4096, 4096] x
// 14336 906 / 865, [8192, 8192] x 8192 1787 / 1741; 16 experts of 1408, 2048 wide, 256 and 1024 rows each, 518 / 485 and 1052 / 1025.
// Bound by their weights, 32 experts of 2048, 7168 wide, 256 rows each: 3770 / 3877.
bool bw_keeps(const mxl_linear& p, int64_t codes) { return codes <= (int64_t)256 << 20 || p.rows >= 512 * (p.groups > 0 ? p.groups : 1); }

int bw_forward(const Linear& l, const void* x, const void* w, const int64_t* lens, void* scratch, void* y, void* stream) {
    const mxl_linear& p = l.p;
    Arena a(scratch);
    const BwForward f(l, a);
    const int fmt = (int)p.act_fmt;
    const bool keep = bw_keeps(p, p.rows * p.k + l.batch * p.n * p.k);
    const mxl::BwTensor in[2] = {{x, p.rows, p.k, 0, nullptr, 0, f.x.q, f.x.s, nullptr, nullptr, keep},
                                 {w, p.n, p.k, l.batch, nullptr, 0, f.w.q, f.w.s, nullptr, nullptr, keep}};
    MXL_TRY(mxl::bw_quantize(in, 2, fmt, stream));
    if (p.groups) return mxl_grouped_gemm_nt_blockwise(f.x.q, f.x.s, fmt, f.w.q, f.w.s, fmt, y, lens, (int)p.groups, p.rows, p.n, p.k, stream);
    return mxl_gemm_nt_blockwise(f.x.q, f.x.s, fmt, f.w.q, f.w.s, fmt, 128, y, p.rows, p.n, p.k, stream);
}

int bw_backward(const Linear& l, int parts, const void* dy, const void* x, const void* w, const int64_t* lens, void* scratch, void* dx, void* dw,
                void* stream) {
    const mxl_linear& p = l.p;
    Arena a(scratch);
    const BwBackward b(l, a);
    const int fmt = (int)p.grad_fmt, G = (int)p.groups;
    if ((parts & MXL_LINEAR_QUANTIZE) && (p.need_dx || p.need_dw)) {
        if (!dy || (p.need_dw && !x) || (p.need_dx && !w)) return MXL_EINVAL;
        mxl::BwTensor in[3];
        int count = 0;
        const bool keep = bw_keeps(p, (p.need_dx ? p.rows * p.n + l.batch * p.k * p.n : 0) + (p.need_dw ? (p.n + p.k) * l.width : 0));
        in[count++] = {dy, p.rows, p.n, 0, p.need_dw ? lens : nullptr, p.need_dw ? G : 0, b.d_row.q, b.d_row.s, b.d_col.q, b.d_col.s, keep};
        if (p.need_dw) in[count++] = {x, p.rows, p.k, 0, lens, G, nullptr, nullptr, b.x_col.q, b.x_col.s, keep};
        if (p.need_dx) in[count++] = {w, p.n, p.k, l.batch, nullptr, 0, nullptr, nullptr, b.w_col.q, b.w_col.s, keep};
        MXL_TRY(mxl::bw_quantize(in, count, fmt, stream));
    }
    if ((parts & MXL_LINEAR_DX) && p.need_dx) {
        if (G) MXL_TRY(mxl_grouped_gemm_nt_blockwise(b.d_row.q, b.d_row.s, fmt, b.w_col.q, b.w_col.s, fmt, dx, lens, G, p.rows, p.k, p.n, stream));
        else MXL_TRY(mxl_gemm_nt_blockwise(b.d_row.q, b.d_row.s, fmt, b.w_col.q, b.w_col.s, fmt, 128, dx, p.rows, p.k, p.n, stream));
    }
    if ((parts & MXL_LINEAR_DW) && p.need_dw) {
        if (G) return mxl_grouped_gemm_wgrad_blockwise(b.d_col.q, b.d_col.s, fmt, b.x_col.q, b.x_col.s, fmt, dw, lens, G, p.rows, p.n, p.k, stream);
        return mxl_gemm_nt_blockwise(b.d_col.q, b.d_col.s, fmt, b.x_col.q, b.x_col.s, fmt, 1, dw, p.n, p.k, l.width, stream);
    }
    return MXL_OK;
}

}  // namespace

extern "C" int mxl_linear_sizes(mxl_linear* p) {
    if (!valid(p)) return MXL_EINVAL;
    const Linear l(p);
    Arena s(nullptr), f(nullptr), b(nullptr);
    if (l.blockwise()) {
        BwForward fwd(l, f);
        BwBackward bwd(l, b);
        p->saved_bytes = 0;
        p->fwd_bytes = f.used;
        p->bwd_bytes = b.used;
        return MXL_OK;
    }
    Saved saved(l, s);
    ForwardScratch fwd(l, f);
    BackwardScratch bwd(l, b);
    p->saved_bytes = s.used;
    p->fwd_bytes = f.used;
    p->bwd_bytes = b.used;
    return MXL_OK;
}

extern "C" int mxl_linear_forward(const mxl_linear* p, const void* x, const void* aux0, const void* aux1, const void* w,
                                  const void* w_scales, const int64_t* lens, void* saved_buf, void* scratch, void* y,
                                  void* stream) {
    if (!valid(p) || !x || !w || !scratch || !y || (p->saved_bytes > 0 && !saved_buf)) return MXL_EINVAL;
    const Linear l(p);
    if (l.blockwise()) return bw_forward(l, x, w, lens, scratch, y, stream);
    const int G = (int)p->groups, batch = (int)l.batch;
    Arena sa(saved_buf), fa(scratch);
    const Saved sv(l, sa);
    const ForwardScratch f(l, fa);
    const int af = (int)p->act_fmt, wf = (int)p->w_fmt;
    const bool from_rows = p->need_dx && p->dx_from_rows;
    const Copy wr = from_rows ? sv.w_row : f.w_row;
    const bool rht = p->rht_signs >= 0 && p->need_dw && p->input == MXL_LINEAR_PLAIN && !l.tensorwise();
    // (a tensor-wise scaled row-wise copy by itself knows no groups, nor do the copies of an input that an RMSNorm forms)
    const bool ungrouped = (l.tensorwise() && !p->need_dw) || p->input == MXL_LINEAR_RMSNORM;
    const mxl::LinearOperands both = {x, w, p->rows, l.batch, p->n, p->k, l.k_ld, l.n_ld, l.w_rows(), ungrouped ? nullptr : lens, ungrouped ? 0 : G,
                                      af, wf, (int)p->scale_mode, l.qf() | (rht ? MXL_QF_RHT_COL : 0u), rht ? (uint32_t)p->rht_signs : 0u, l.keeps(),
                                      f.x_amax, f.w_amax, sv.x_si, sv.w_si,
                                      p->input == MXL_LINEAR_RMSNORM ? aux0 : nullptr, sv.rstd,
                                      f.x_row.q, f.x_row.s, sv.x_col.q, sv.x_col.s, wr.q, wr.s, sv.w_col.q, sv.w_col.s};
    auto product = [&](const Copy& wc, const float* alpha_a, const float* alpha_b) {
        return mxl::gemm_nt_held(f.x_row.q, f.x_row.s, af, wc.q, wc.s, wf, y, lens, batch, p->rows, p->n, l.k_ld, alpha_a, alpha_b, MXL_GF_KSTEP, nullptr,
                                 stream, l.w_rows(), true);
    };
    if (l.tensorwise()) {
        MXL_TRY(mxl::amax_pair(x, p->rows * p->k, f.x_amax, w, l.batch * p->n * p->k, f.w_amax, true, stream));
        MXL_TRY(mxl::quantize_pair(both, stream));
        return product(wr, sv.x_si, sv.w_si);
    }
    if (p->input == MXL_LINEAR_RMSNORM) {
        MXL_TRY(mxl_rmsnorm_fwd(x, aux0, (float)p->eps, p->rows, p->k, nullptr, sv.rstd, stream));
        if (!p->w_quantized && G == 0 && aux0) {
            MXL_TRY(mxl::quantize_pair(both, stream));
            return product(wr, nullptr, nullptr);
        }
        if (!aux0 || !sv.rstd) return MXL_EINVAL;
        mxl::LinearInput in{x};
        in.norm_w = aux0;
        in.rstd = sv.rstd;
        MXL_TRY(mxl::quantize_input(in, p->rows, p->k, l.k_ld, af, (int)p->scale_mode, nullptr, 0, f.x_row.q, f.x_row.s, sv.x_col.q, sv.x_col.s, l.qf(), 0,
                                    0, l.keeps(), stream));
    } else if (p->input != MXL_LINEAR_PLAIN) {
        if (!aux0 || (p->probs_dtype != MXL_PROBS_F32 && p->probs_dtype != MXL_PROBS_BF16)) return MXL_EINVAL;
        mxl::LinearInput in{x};
        in.act = p->input == MXL_LINEAR_SILU ? MXL_ACT_SILU : MXL_ACT_GELU;
        in.probs = aux0;
        in.probs_dtype = (int)p->probs_dtype;
        in.row_mask = (const uint8_t*)aux1;
        MXL_TRY(mxl::quantize_input(in, p->rows, p->k, l.k_ld, af, (int)p->scale_mode, lens, G, f.x_row.q, f.x_row.s, sv.x_col.q, sv.x_col.s, l.qf(), 0, 0,
                                    l.keeps(), stream));
    } else if (!p->w_quantized) {
        MXL_TRY(mxl::quantize_pair(both, stream));
        return product(wr, nullptr, nullptr);
    } else {
        MXL_TRY(mxl::quantize_input({x}, p->rows, p->k, l.k_ld, af, (int)p->scale_mode, lens, G, f.x_row.q, f.x_row.s, sv.x_col.q, sv.x_col.s, both.flags, 0,
                                    both.rht_signs, l.keeps(), stream));
    }
    if (p->w_quantized) {
        if (!w_scales) return MXL_EINVAL;
        return mxl_grouped_gemm_nt_ex(f.x_row.q, f.x_row.s, af, w, w_scales, wf, y, lens, batch, p->rows, p->n, l.k_ld, MXL_GF_KSTEP, stream);
    }
    MXL_TRY(mxl::quantize_weight_rows(w, l.batch, p->n, p->k, l.k_ld, l.n_ld, l.w_rows(), wf, (int)p->scale_mode, wr.q, wr.s, sv.w_col.q, sv.w_col.s,
                                      l.qf(), l.keeps(), stream));
    return product(wr, nullptr, nullptr);
}

extern "C" int mxl_linear_backward(const mxl_linear* p, int parts, const void* dy, const void* x, const void* aux0, const void* aux1,
                                   const void* wt, const void* wt_scales, const int64_t* lens, void* saved_buf, void* scratch, void* dx,
                                   void* daux, void* dw, uint32_t dw_flags, uint64_t sr_seed, void* stream) {
    if (!valid(p) || !scratch || (dw_flags & ~(uint32_t)MXL_GF_ACCUM_F32)) return MXL_EINVAL;
    const Linear l(p);
    if (l.blockwise()) return dw_flags ? MXL_EINVAL : bw_backward(l, parts, dy, x, wt, lens, scratch, dx, dw, stream);
    const int G = (int)p->groups, batch = (int)l.batch;
    Arena sa(saved_buf), ba(scratch);
    const Saved sv(l, sa);
    const BackwardScratch b(l, ba);
    const int gf = (int)p->grad_fmt, wf = (int)p->w_fmt;
    const bool sr = p->grad_sr && gf == MXL_FMT_E2M1;
    const bool dx_part = (parts & MXL_LINEAR_DX) && p->need_dx, dw_part = (parts & MXL_LINEAR_DW) && p->need_dw;
    // Experts bound by their weights: dgrad reads those, a gigabyte perhaps, and leaves nothing in the cache of what the weight gradient reads.
    // So that one goes first and finds the gradient's transposed copy there.  us a pass: 32 experts of 2048, 7168 wide, 256 rows each, 2719 ->
    // 2692 (the order alone 2707, the copies kept alone 2740), E2M1 2036 -> 1994; 8 experts of 14336, 4096 wide, 256 rows each, E2M1 2007 ->
    // 1950, FP8 2681 -> 2672; no difference with 16 experts of 4096, 4096 wide.  (Dense gradients this small share a launch, below.)
    // dgrad's operands are looked at before either is launched: a call that it refuses has added nothing to a weight gradient.
    const bool dw_first = dw_part && dx_part && p->groups > 0 && l.mx() && !l.keeps();
    if (parts & MXL_LINEAR_QUANTIZE) {
        if (!dy) return MXL_EINVAL;
        if (l.tensorwise()) {
            MXL_TRY(mxl::amax_pair(dy, p->rows * p->n, b.amax, nullptr, 0, nullptr, true, stream));
            MXL_TRY(mxl::quantize_tensorwise_parts(dy, p->rows, p->n, p->need_dx ? l.n_ld : 0, gf, b.amax, p->need_dw ? lens : nullptr, p->need_dw ? G : 0,
                                            b.d_row.q, b.d_row.s, b.d_col.q, b.d_col.s, b.d_si, l.qf(), stream));
        } else {
            const bool rht = p->rht_signs >= 0 && p->need_dw;
            MXL_TRY(mxl::quantize_input({dy}, p->rows, p->n, l.n_ld, gf, (int)p->scale_mode, lens, G, b.d_row.q, b.d_row.s, b.d_col.q, b.d_col.s,
                                        l.qf() | (rht ? MXL_QF_RHT_COL : 0u) | (sr ? MXL_QF_SR : 0u), sr ? sr_seed : 0,
                                        rht ? (uint32_t)p->rht_signs : 0u, l.keeps() || dw_first, stream));
        }
    }
    // the two GEMMs: where both run on small tiles, in one launch
    mxl::HeldGemm hold;
    hold.behind = dw_first;
    if (dx_part) {
        void* out = b.dxi ? b.dxi : dx;
        if (!out) return MXL_EINVAL;
        const uint32_t flags = MXL_GF_KSTEP | (p->dx_from_rows ? MXL_GF_B_TRANSPOSED : 0u);
        const void* bq = p->w_quantized ? wt : p->dx_from_rows ? sv.w_row.q : sv.w_col.q;
        const void* bs = p->w_quantized ? wt_scales : sv.w_col.s;
        const bool tw = l.tensorwise();
        if (tw && (!b.d_si || !sv.w_si)) return MXL_EINVAL;
        MXL_TRY(mxl::gemm_nt_held(b.d_row.q, b.d_row.s, gf, bq, bs, wf, out, lens, batch, p->rows, p->k, l.n_ld, tw ? b.d_si : nullptr,
                                  tw ? sv.w_si : nullptr, flags, dw_part ? &hold : nullptr, stream));
    }
    int rc = MXL_OK;
    if (dw_part) {
        const bool tw = l.tensorwise();
        if (tw && (!b.d_si || !sv.x_si)) rc = MXL_EINVAL;
        else
            rc = mxl::gemm_wgrad_held(b.d_col.q, b.d_col.s, gf, sv.x_col.q, sv.x_col.s, (int)p->act_fmt, dw, lens, G, p->rows, p->n, p->k,
                                      tw ? b.d_si : nullptr, tw ? sv.x_si : nullptr, MXL_GF_KSTEP | dw_flags, dw_first ? nullptr : &hold, stream);
    }
    MXL_TRY(hold.flush((hipStream_t)stream));
    MXL_TRY(rc);
    if (dx_part) {
        if (p->input == MXL_LINEAR_RMSNORM)
            MXL_TRY(mxl_rmsnorm_bwd(b.dxi, x, aux0, sv.rstd, p->rows, p->k, dx, daux, b.norm_ws, b.norm_bytes, stream));
        else if (p->input != MXL_LINEAR_PLAIN)
            MXL_TRY(mxl::glu_probs_bwd(b.dxi, x, aux0, (int)p->probs_dtype, (const uint8_t*)aux1, p->rows, p->k,
                                       p->input == MXL_LINEAR_SILU ? MXL_ACT_SILU : MXL_ACT_GELU, dx, daux, p->need_dw && !dw_part, stream));
    }
    return MXL_OK;
}
