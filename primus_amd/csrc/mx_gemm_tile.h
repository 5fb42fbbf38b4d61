// Entry points of the small-tile GEMM kernel (mx_gemm_tile.hip, mx_gemm_pair.hip) for the dispatch in mx_gemm.hip.
#pragma once
#include "mx_gemm_choice.h"
#include "mx_gemm_common.h"

namespace mxl {

// A dense weight gradient over few tokens runs the 128 x 128 tile with two stages instead of four: more workgroups on a
// CU overlap their outputs (1024 tokens, 14336 x 4096: 69 -> 64 us, 256 tokens 35 -> 29; 2048 tokens, 4096 x 4096: 33 -> 40).
inline bool tile_wgrad_shallow(const GemmArgs& a) { return a.k / a.num_groups <= 1024; }

// Operands and formats as the ring kernel takes them (K-step-major, at most 256 groups, no fp32 accumulation).
int gemm_tile_fwd(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);
int gemm_tile_wgrad(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);
int gemm_tile_bt(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st);
// the ring kernel, forward / dgrad, on operands that the dispatch has looked at
int gemm_ring_fwd(bool bt, int afmt, int bfmt, const GemmArgs& a, int64_t max_tiles, hipStream_t st);

// A linear's input gradient, prepared and not yet launched: where the weight gradient that follows runs on small tiles
// too, both go in one launch (mx_gemm_pair.hip).  `behind`: it is put off whatever it runs on, and launched behind the weight gradient.
// Lives on the stack of the call that launches both.
struct HeldGemm {
    bool held = false, behind = false, bt;
    int afmt, bfmt, tile;
    int64_t max_tiles;
    GemmArgs args;
    // the input gradient in a launch of its own, if it is still held
    int flush(hipStream_t st) {
        if (!held) return MXL_OK;
        held = false;
        if (tile == TILE_RING) return gemm_ring_fwd(bt, afmt, bfmt, args, max_tiles, st);
        return bt ? gemm_tile_bt(afmt, bfmt, args, tile, st) : gemm_tile_fwd(afmt, bfmt, args, tile, st);
    }
};
// is there a launch for this input gradient together with a weight gradient?
bool gemm_pair_takes(const HeldGemm& h);
// both; the weight gradient's rows are the input gradient's, in the same format, and its columns E4M3 (E2M1 with E2M1 rows)
int gemm_pair(const HeldGemm& h, const GemmArgs& wgrad, hipStream_t st);

// mxl_grouped_gemm_nt_ex / _scaled and mxl_grouped_gemm_wgrad_ex / _scaled (alpha null or given), with the former put off
// into `hold` if it runs on small tiles (or hold->behind), and the latter launched with what is held.  b_rows: rows from one group's matrix in b
// to the next (0: n); b_fresh: the caller has just quantised b
int gemm_nt_held(const void* a_codes, const void* a_scales, int a_fmt, const void* b_codes, const void* b_scales, int b_fmt, void* c,
                 const int64_t* group_lens, int num_groups, int64_t total_m, int64_t n, int64_t k, const float* alpha_a,
                 const float* alpha_b, uint32_t flags, HeldGemm* hold, void* stream, int64_t b_rows = 0, bool b_fresh = false);
int gemm_wgrad_held(const void* a_codes, const void* a_scales, int a_fmt, const void* b_codes, const void* b_scales, int b_fmt, void* c,
                    const int64_t* group_lens, int num_groups, int64_t total_m, int64_t n, int64_t k, const float* alpha_a,
                    const float* alpha_b, uint32_t flags, HeldGemm* hold, void* stream);

}  // namespace mxl
