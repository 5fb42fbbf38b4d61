// The GEMMs on small output tiles as launches of their own; two of them in one launch: mx_gemm_pair.hip.
#include "mx_gemm_tile_body.h"

namespace mxl {

template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT, int TM, int TN, int ST>
__global__ __launch_bounds__(256, 2) void mx_gemm_tile_kernel(GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    gemm_tile_body<AFMT, BFMT, MODE, ALPHA, BT, TM, TN, ST>(p, blockIdx.x, smem);
}

template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT, int TM, int TN, int ST>
static int launch_tile(const GemmArgs& a, hipStream_t st) {
    constexpr int lds = tile_lds_bytes<TM, TN, ST>(BFMT == kFmtE2M1 && AFMT != kFmtE2M1);
    static std::atomic<bool> attr_set[64];
    return launch_tiles(mx_gemm_tile_kernel<AFMT, BFMT, MODE, ALPHA, BT, TM, TN, ST>, attr_set, lds, tile_grid<MODE, TM, TN>(a), st, a);
}

// Forward and input gradients: eight stages where every CU has at most one workgroup and its contraction is at least 48 K
// steps long, else four.  Alone on its CU a workgroup waits for memory at the distance it asks ahead: a K step's MFMAs are
// over in a quarter of a microsecond, and with four stages 224 CUs keep 5 MB on their way, which over the latency is half of
// what the memory delivers.
// us, four / eight stages, weights from memory: 64 x 64 tiles, [64, 4096] x 14336 16.8 / 13.7, [64, 14336] x 4096 44.2 / 31.4,
// [32, 8192] x 8192 28.8 / 19.4, [256, 4096] x 4096 10.6 / 8.5; with more than 256 tiles [512, 4096] x 4096 13.8 / 14.3.
// 64 x 128 tiles, [512, 4096] x 4096 13.3 / 12.3; E2M1 weights against FP8 rows, [64, 4096] x 14336 14.5 / 11.5.
// Shorter ranges lose a little where the weights are in the cache (32 steps, 8 groups of 25 rows, [1024, 2048], 7.5 / 7.9), and
// so do 128 x 128 tiles, which have more to do in a step ([512, 4096] x 4096 14.8 / 15.1).
constexpr int64_t STAGE_CUS = 256, STAGE_STEPS = 48;
template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT, int TM, int TN>
static int launch_staged(const GemmArgs& a, hipStream_t st) {
    if constexpr (MODE == MODE_FWD) {
        constexpr int64_t step = AFMT == kFmtE2M1 ? 2 * BK : BK;
        if (a.k >= STAGE_STEPS * step && tile_grid<MODE, TM, TN>(a) <= STAGE_CUS) return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, TM, TN, 8>(a, st);
    }
    return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, TM, TN, 4>(a, st);
}

template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT>
static int pick_tile(const GemmArgs& a, int tile, hipStream_t st) {
    if constexpr (!BT) {
        if (tile == TILE_64) return launch_staged<AFMT, BFMT, MODE, ALPHA, BT, 64, 64>(a, st);
    }
    if (tile == TILE_64 || tile == TILE_64x128) return launch_staged<AFMT, BFMT, MODE, ALPHA, BT, 64, 128>(a, st);
    if constexpr (MODE == MODE_WGRAD) {
        if (tile_wgrad_shallow(a)) return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, 128, 128, 2>(a, st);
    }
    return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, 128, 128, 4>(a, st);
}

template <int MODE>
static int by_format(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st) {
    if (a.alpha_a != nullptr) {
        if (afmt == MXL_FMT_E5M2 && bfmt == MXL_FMT_E5M2) return pick_tile<MXL_FMT_E5M2, MXL_FMT_E5M2, MODE, true, false>(a, tile, st);
        if (afmt == MXL_FMT_E5M2) return pick_tile<MXL_FMT_E5M2, MXL_FMT_E4M3, MODE, true, false>(a, tile, st);
        return pick_tile<MXL_FMT_E4M3, MXL_FMT_E4M3, MODE, true, false>(a, tile, st);
    }
    if (afmt == MXL_FMT_E2M1) return pick_tile<MXL_FMT_E2M1, MXL_FMT_E2M1, MODE, false, false>(a, tile, st);
    if constexpr (MODE == MODE_FWD) {
        if (bfmt == MXL_FMT_E2M1) return pick_tile<MXL_FMT_E4M3, MXL_FMT_E2M1, MODE_FWD, false, false>(a, tile, st);
    }
    return pick_tile<MXL_FMT_E4M3, MXL_FMT_E4M3, MODE, false, false>(a, tile, st);
}

int gemm_tile_fwd(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st) { return by_format<MODE_FWD>(afmt, bfmt, a, tile, st); }
int gemm_tile_wgrad(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st) { return by_format<MODE_WGRAD>(afmt, bfmt, a, tile, st); }
int gemm_tile_bt(int afmt, int bfmt, const GemmArgs& a, int tile, hipStream_t st) {
    if (bfmt == MXL_FMT_E2M1) return pick_tile<MXL_FMT_E2M1, MXL_FMT_E2M1, MODE_FWD, false, true>(a, tile, st);
    if (a.alpha_a == nullptr) return pick_tile<MXL_FMT_E4M3, MXL_FMT_E4M3, MODE_FWD, false, true>(a, tile, st);
    if (afmt == MXL_FMT_E5M2) return pick_tile<MXL_FMT_E5M2, MXL_FMT_E4M3, MODE_FWD, true, true>(a, tile, st);
    return pick_tile<MXL_FMT_E4M3, MXL_FMT_E4M3, MODE_FWD, true, true>(a, tile, st);
}

}  // namespace mxl
