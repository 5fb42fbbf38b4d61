// A linear's input gradient and weight gradient on small tiles in one launch.
//
// Over a few hundred tokens neither fills the chip for long: the input gradient of [256, 4096] x [4096, 4096] is 128 tiles
// of 64 K steps, the weight gradient 1024 tiles of four, and one after the other they leave the CUs idle at the end of
// each.  A whole pass of that linear as a graph: 80 us with two launches, 73 so; linear 1999 x 2880 -> 5760, forward +
// backward, 173 -> 158 us (both gradients on 128 x 128 tiles, three rounds each of 720 and 1035).  Here the workgroups of the input gradient, which run longest, come first and the weight gradient's
// fill up behind them.  Each tile is the body of mx_gemm_tile.hip, so the bits are the same.
#include "mx_gemm_tile_body.h"
#include "mx_gemm_tile.h"

namespace mxl {

// FMT: format of the gradient, WFMT: of the weight and the activation; TM1 x 128 tiles for the input gradient, 128 x 128
// with ST2 stages for the weight gradient
template <int FMT, int WFMT, bool ALPHA, bool BT, int TM1, int ST2>
__global__ __launch_bounds__(256, 2) void mx_gemm_pair_kernel(GemmArgs d, GemmArgs w, uint32_t first) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    if (blockIdx.x < first) gemm_tile_body<FMT, WFMT, MODE_FWD, ALPHA, BT, TM1, 128, 4>(d, blockIdx.x, smem);
    else gemm_tile_body<FMT, WFMT, MODE_WGRAD, ALPHA, false, 128, 128, ST2>(w, blockIdx.x - first, smem);
}

template <int FMT, int WFMT, bool ALPHA, bool BT, int TM1, int ST2>
static int launch_pair(const GemmArgs& d, const GemmArgs& w, hipStream_t st) {
    constexpr int l1 = tile_lds_bytes<TM1, 128, 4>(false), l2 = tile_lds_bytes<128, 128, ST2>(false);
    static std::atomic<bool> attr_set[64];
    const int64_t first = tile_grid<MODE_FWD, TM1, 128>(d);      // a multiple of 8: the weight gradient's keep their XCDs
    return launch_tiles(mx_gemm_pair_kernel<FMT, WFMT, ALPHA, BT, TM1, ST2>, attr_set, l1 > l2 ? l1 : l2, first + tile_grid<MODE_WGRAD, 128, 128>(w),
                        st, d, w, (uint32_t)first);
}

template <int FMT, int WFMT, bool ALPHA, bool BT>
static int pick_pair(const HeldGemm& h, const GemmArgs& w, hipStream_t st) {
    const bool shallow = tile_wgrad_shallow(w);
    if (h.tile == TILE_128) return shallow ? launch_pair<FMT, WFMT, ALPHA, BT, 128, 2>(h.args, w, st) : launch_pair<FMT, WFMT, ALPHA, BT, 128, 4>(h.args, w, st);
    return shallow ? launch_pair<FMT, WFMT, ALPHA, BT, 64, 2>(h.args, w, st) : launch_pair<FMT, WFMT, ALPHA, BT, 64, 4>(h.args, w, st);
}

bool gemm_pair_takes(const HeldGemm& h) {
    if (h.tile != TILE_128 && h.tile != TILE_64x128) return false;
    if (h.args.alpha_a != nullptr) return h.afmt == MXL_FMT_E5M2 && h.bfmt == MXL_FMT_E4M3;
    return h.afmt == h.bfmt && h.afmt != MXL_FMT_E5M2;
}

int gemm_pair(const HeldGemm& h, const GemmArgs& w, hipStream_t st) {
    if (h.args.alpha_a != nullptr)
        return h.bt ? pick_pair<MXL_FMT_E5M2, MXL_FMT_E4M3, true, true>(h, w, st) : pick_pair<MXL_FMT_E5M2, MXL_FMT_E4M3, true, false>(h, w, st);
    if (h.afmt == MXL_FMT_E2M1)
        return h.bt ? pick_pair<MXL_FMT_E2M1, MXL_FMT_E2M1, false, true>(h, w, st) : pick_pair<MXL_FMT_E2M1, MXL_FMT_E2M1, false, false>(h, w, st);
    return h.bt ? pick_pair<MXL_FMT_E4M3, MXL_FMT_E4M3, false, true>(h, w, st) : pick_pair<MXL_FMT_E4M3, MXL_FMT_E4M3, false, false>(h, w, st);
}

}  // namespace mxl
