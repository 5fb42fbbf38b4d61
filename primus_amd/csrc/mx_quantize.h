// Both operands of a linear's forward, quantised (mx_quantize.hip) for the calls in mx_linear.hip.
#pragma once
#include <stdint.h>

namespace mxl {

// An abs-max launch leaves one value per workgroup (amax_parts(n) of them for n elements), at most this many.
constexpr int AMAX_PARTS = 512;
int amax_parts(int64_t n);
int amax_pair(const void* a, int64_t na, void* out_a, const void* b, int64_t nb, void* out_b, bool parts, void* stream);
// mxl_quantize_tensorwise on such parts of x
int quantize_tensorwise_parts(const void* x, int64_t rows, int64_t cols, int64_t row_ld, int fmt, const float* amax, const int64_t* group_lens,
                              int num_groups, void* q_row, void* s_row, void* q_colT, void* s_colT, float* scale_inv, uint32_t flags,
                              void* stream);

struct LinearOperands {
    // activations [rows, k] (ragged groups: group_lens, num_groups; 0 and null: one), weights [batch, n, k]
    const void *x, *w;
    int64_t rows, batch, n, k, k_ld, n_ld;
    int64_t w_rows;                     // rows per matrix of the weight's row-wise copy: n, or n_ld with zeros behind the n
    const int64_t* group_lens;
    int num_groups;
    int x_fmt, w_fmt, scale_mode;
    uint32_t flags, rht_signs;          // MXL_QF_* of mxl_quantize_ex (no stochastic rounding)
    bool keep;                          // codes that fit the caches are stored through them
    // tensor-wise scaling: abs-max of each on the device (the parts of amax_pair), and where 1 / scale goes; null otherwise
    const float *x_amax, *w_amax;
    float *x_scale_inv, *w_scale_inv;
    // the input an RMSNorm forms from x, its weight and the rows' statistics (mxl_rmsnorm_fwd); null: x itself
    const void *norm_w, *rstd;
    // the copies; transposed ones may be null as mxl_quantize_ex and mxl_quantize_weight_2d_ex allow
    uint8_t *xq_row, *xs_row, *xq_col, *xs_col, *wq_row, *ws_row, *wq_col, *ws_col;
};
// in one launch where there is a kernel for the two, else one after the other; the same bytes
int quantize_pair(const LinearOperands& o, void* stream);
// mxl_quantize_weight_2d_ex with `rows` rows per matrix in the row-wise copy
int quantize_weight_rows(const void* w, int64_t batch, int64_t n, int64_t k, int64_t k_ld, int64_t n_ld, int64_t rows, int fmt, int scale_mode,
                         void* q_row, void* s_row, void* q_colT, void* s_colT, uint32_t flags, bool keep, void* stream);

// One operand that is quantised by itself: x as it is, what a gated activation turns it into (act, probs, probs_dtype, row_mask),
// or what an RMSNorm does (norm_w, rstd)
struct LinearInput {
    const void* x;
    int act = -1;                       // MXL_ACT_*
    const void* probs = nullptr;
    int probs_dtype = 0;
    const uint8_t* row_mask = nullptr;
    const void *norm_w = nullptr, *rstd = nullptr;
};
// mxl_quantize_ex, mxl_glu_probs_quantize, mxl_rmsnorm_quantize with `keep`
int quantize_input(const LinearInput& o, int64_t rows, int64_t cols, int64_t row_ld, int fmt, int scale_mode, const int64_t* group_lens, int num_groups,
                   void* q_row, void* s_row, void* q_colT, void* s_colT, uint32_t flags, uint64_t sr_seed, uint32_t rht_signs, bool keep, void* stream);

}  // namespace mxl
