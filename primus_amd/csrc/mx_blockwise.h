// Several tensors quantised under the 128-blockwise recipe in one launch (mx_blockwise.hip), for the calls in mx_linear.hip.
#pragma once
#include <stdint.h>

namespace mxl {

struct BwTensor {
    const void* x;                 // activation [rows, cols], or a batch of weights [batch, rows, cols]
    int64_t rows, cols;
    int64_t batch;                 // 0: an activation
    const int64_t* group_lens;     // activations only; null: one group
    int num_groups;
    void *q_row, *sinv_row, *q_colT, *sinv_colT;
    bool keep;                     // codes are stored through the caches instead of past them
};
// 1 to 3 tensors of one format, as mxl_quantize_blockwise and mxl_quantize_blockwise_weight take them
int bw_quantize(const BwTensor* tensors, int count, int fmt, void* stream);

}  // namespace mxl
