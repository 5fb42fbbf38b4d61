// mxl_glu_probs_bwd for the calls in mx_linear.hip, which know what else is running.
#pragma once
#include <stdint.h>

namespace mxl {

int glu_probs_bwd(const void* dy_bf16, const void* x_bf16, const void* probs, int probs_dtype, const uint8_t* row_mask, int64_t rows, int64_t f, int act,
                  void* dx_bf16, void* dprobs_f32, bool shared, void* stream);

}  // namespace mxl
