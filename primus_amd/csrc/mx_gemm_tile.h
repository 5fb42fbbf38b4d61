// Entry points of the small-tile GEMM kernel (mx_gemm_tile.hip) for the dispatch in mx_gemm.hip.
#pragma once
#include "mx_gemm_common.h"

namespace mxl {

enum { TILE_RING = 0, TILE_64 = 1, TILE_64x128 = 2, TILE_128 = 3 };

// A dense weight gradient over few tokens runs the 128 x 128 tile with two stages instead of four: more workgroups on a
// CU overlap their outputs (1024 tokens, 14336 x 4096: 69 -> 64 us, 256 tokens 35 -> 29; 2048 tokens, 4096 x 4096: 33 -> 40).
inline bool tile_wgrad_shallow(const GemmArgs& a) { return a.k / a.num_groups <= 1024; }

// Operands and formats as the ring kernel takes them (K-step-major, at most 256 groups, no fp32 accumulation).
int gemm_tile_fwd(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);
int gemm_tile_wgrad(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);
int gemm_tile_bt(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);

}  // namespace mxl
