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

template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT>
static int pick_tile(const GemmArgs& a, int tile, hipStream_t st) {
    if constexpr (!BT) {
        if (tile == TILE_64) return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, 64, 64, 4>(a, st);
    }
    if (tile == TILE_64 || tile == TILE_64x128) return launch_tile<AFMT, BFMT, MODE, ALPHA, BT, 64, 128, 4>(a, st);
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
