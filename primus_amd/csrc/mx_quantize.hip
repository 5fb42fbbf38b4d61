// MX quantisers for gfx950: bf16 -> {E4M3, E2M1} codes + E8M0 block scales.
//
// One kernel family covers the three layouts the linear path needs
// (primus_turbo.py:321-354, primus_turbo_mxfp4_local.py:147-207):
//   ROW  : blocks of 32 along the columns, output in the input's orientation;
//   COL  : blocks of 32 along the rows, output TRANSPOSED, blocks restarting at
//          every expert boundary, each expert segment padded to 128;
//   TWOD : one scale per 32x32 tile (weights), both copies from one scale.
//
// A workgroup (256 threads, 4 waves) owns a 128x128 tile.  Wave w owns rows
// [32w, 32w+32) -- exactly one column-wise MX block -- and each lane loads
// 8 rows x 8 columns as eight 16-byte loads, so a 16-lane group reads 256
// contiguous bytes.  Row-block maxima are reduced over 4 adjacent lanes with
// DPP, column-block maxima in registers over the lane's 8 rows and then over
// the 4 lane groups.  The transposed codes go through an LDS tile so that the
// global stores are 128 contiguous bytes per output row.
#include "mx_device.h"
#include "mx_quantize.h"

namespace mxl {

constexpr int QT = 128;       // tile edge
constexpr int QTHREADS = 256;
constexpr int AMAX_MAX_WG = AMAX_PARTS;     // workgroups of an abs-max launch per tensor

struct QuantArgs {
    const uint16_t* x;
    int64_t rows, cols;
    const int64_t* group_lens;
    int num_groups;
    uint8_t* q_row;
    uint8_t* s_row;
    uint8_t* q_colT;
    uint8_t* s_colT;
    int64_t row_ld;     // columns of the row-wise copy (>= cols; the excess is zero-filled padding)
    int64_t W;          // padded width of the transposed copy (elements)
    int64_t mat_rows;   // TWOD: rows per matrix (n); otherwise unused
    int64_t out_rows;   // TWOD: rows per matrix in the row-wise copy, n or n rounded up to whole tiles (the excess is written as zeros)
    // fused gated activation in front (ACT >= 0): x is fc1's output [rows, 2 * cols], the tensor that is
    // quantised is act(x[:, :cols]) * x[:, cols:] * probs[row], masked rows are zero
    const void* probs;
    int probs_bf16;
    const uint8_t* row_mask;
    // fused RMSNorm in front (ACT == PRO_RMSNORM): the tensor that is quantised is (x * rstd[row]) * norm_w[col];
    // rstd travels in `probs` (fp32)
    const uint16_t* norm_w;
    // tensor-wise scaling (SMODE == SCALE_TENSOR): one fp32 scale for the whole tensor, fp8_max / max(amax, 1e-12),
    // from the tensor's abs-max on the device; its reciprocal is written to scale_inv_out (may be null).  The
    // block-scale arrays are filled with 127 (2^0), so the scaled GEMM reads the codes unchanged.
    const float* tensor_amax;
    int amax_parts;         // number of values at tensor_amax, whose maximum it is
    float* scale_inv_out;
    // Code layout of both copies.  0: row-major [rows, ld].  1: K-chunk-major [ld / 128][rows][128 elements]:
    // the 128 elements of a row that one GEMM K slot consumes stay together and consecutive rows follow
    // each other, so a GEMM tile's slot is one contiguous block and this kernel writes 128 x 128-element
    // pieces contiguously.  chunk_rows_row / chunk_rows_col: rows of the whole row-wise / transposed operand.
    // 2: K-step-major (FP8 only): codes [ld / 64][rows][64], scales [ceil(ld / 512)][rows][16].
    int kchunk;
    int64_t chunk_rows_row, chunk_rows_col;
    uint64_t sr_seed;       // SR kernels: seed of the stochastic rounding
    uint32_t rht_signs;     // RHT kernels: sign bit i flips row i of every 16-row group before the transform
    bool keep_row, keep_col;    // codes are stored through the caches (keep_in_cache)
    int tiles_r, tiles_c;   // tile grid: row tiles (upper bound when grouped) x column tiles
    int super_c, n_super;   // supertiles: count along the columns, total
    int super_log;          // log2 of a supertile's edge in tiles
};

// Workgroup -> tile.  Workgroups are dealt to the 8 XCDs round robin, so workgroup L is the
// (L / 8)-th one of XCD L % 8.  Each XCD walks whole supertiles, column tile fastest:
//  - the pieces of the scale arrays that neighbouring tiles write meet in one L2 and leave it as one write instead
//    of several partial ones: 4 bytes of each of 8 neighbours in the row-major layouts, 2 + 2 bytes of each of 4 in a
//    16-byte panel row;
//  - the workgroups resident at any moment cover long contiguous row spans instead of one 256-byte
//    column slice at a power-of-two stride, which would camp on a few memory channels.
// 4 x 4 tiles with scale panels, 8 x 8 without: the XCDs' shares of a small tensor are the more even the smaller the
// supertile (both copies of [1999, 5760]: 14.7 us on 8 x 8, 12.2 on 4 x 4 and on 2 x 2; [1000, 1024] 8.9, 7.2, 7.3; weight
// [5760, 2880] 15.0, 13.8, 13.9; [8192, 14336] 93.3, 90.3, 91.7).
__device__ __forceinline__ bool quant_tile_of_workgroup(const QuantArgs& a, int L, int& pt, int& ct) {
    const int xcd = L & 7, k = L >> 3;
    const int lg = a.super_log;
    const int s = (k >> (2 * lg)) * 8 + xcd;
    if (s >= a.n_super) return false;
    const int within = k & ((1 << (2 * lg)) - 1);
    pt = ((s / a.super_c) << lg) + (within >> lg);
    ct = ((s % a.super_c) << lg) + (within & ((1 << lg) - 1));
    return pt < a.tiles_r && ct < a.tiles_c;
}

// SR (E2M1 only): codes are rounded stochastically instead of to nearest even; scales are unaffected.
// The random word of a pair of neighbouring elements is a function of the seed and of the pair's
// position in the OUTPUT (row-wise copy: row, column pair; transposed copy: column, position pair
// along the padded token axis), so the result does not depend on the tiling.
//
// RHT: the transposed copy is taken from a randomised Hadamard transform of the input along the token
// axis (colwise_use_rht of quantize_mxfp4_dual, primus_turbo_mxfp4_local.py:234-250,272-288): every
// group of 16 consecutive token positions of an expert's segment becomes (1/4) H16 (s * x), H16 the
// Sylvester matrix and s the sign vector `rht_signs`, evaluated as four fp32 butterfly stages (strides
// 1, 2, 4, 8) and rounded once to bf16; that tensor is then quantised like any other.  The transform is
// orthogonal, so a wgrad GEMM whose two operands were both transformed computes the same contraction
// while single large values are spread over 16 positions before they meet the 4-bit grid.
constexpr int PRO_RMSNORM = 2;   // value of ACT next to MXL_ACT_SILU (0) and MXL_ACT_GELU (1)
constexpr int SCALE_TENSOR = 3;  // value of SMODE next to the three E8M0 rules: per-tensor fp32 scale

template <int FMT, int SMODE> __device__ __forceinline__ uint32_t block_byte(uint32_t amax16) {
    if constexpr (SMODE == SCALE_TENSOR) {
        return 127u;
    } else {
        return scale_byte<FMT, SMODE>(amax16);
    }
}

// K-step-major scales: a row's 16 bytes of a panel (512 elements = 8 MFMA K steps of two blocks) are ordered
// [block parity][K step], so that the 8 bytes a GEMM lane needs for the panel's 8 steps are adjacent (the lanes
// 0-31 of an MFMA supply the scales of the even blocks, the lanes 32-63 those of the odd ones).  `v` = the scale
// bytes of the four blocks of 128-element tile `quarter` of the panel.
__device__ __forceinline__ void store_panel_scales(uint8_t* row16, int quarter, uint32_t v) {
    *(uint16_t*)(row16 + 2 * quarter) = (uint16_t)((v & 0xFFu) | ((v >> 8) & 0xFF00u));
    *(uint16_t*)(row16 + 8 + 2 * quarter) = (uint16_t)(((v >> 8) & 0xFFu) | ((v >> 16) & 0xFF00u));
}

template <int FMT, int SMODE, bool ROW, bool COL, bool TWOD, int ACT = -1, bool SR = false, bool RHT = false>
__device__ __forceinline__ void quant_workgroup(const QuantArgs& a, int block) {
    constexpr bool FP4 = (FMT == kFmtE2M1);
    constexpr bool TENSOR = (SMODE == SCALE_TENSOR);
    static_assert(TENSOR || FMT != kFmtE5M2, "E5M2 exists for tensor-wise scaling only");
    static_assert(!TENSOR || (!FP4 && !SR && !RHT && ACT < 0), "tensor-wise scaling: FP8 codes, plain input");
    static_assert(!SR || (FP4 && !TWOD && ACT < 0), "stochastic rounding exists for 1-D E2M1 quantisation only");
    static_assert(!RHT || (COL && !TWOD && ACT < 0), "the Hadamard transform applies to the transposed 1-D copy only");
    constexpr int TPITCH = FP4 ? (QT / 2 + 16) : (QT + 16);  // bytes per LDS row of the transposed tile
    __shared__ __attribute__((aligned(16))) uint8_t t_tile[COL ? QT * TPITCH : 16];
    __shared__ uint32_t srow_tile[QT];
    __shared__ uint32_t scol_tile[QT];

    const int t = threadIdx.x;
    const int w = t >> 6, l = t & 63, c16 = l & 15, rg = l >> 4;
    // tensor-wise: the abs-max is the maximum of amax_parts values, up to eight to a lane, which every wave takes for itself;
    // they are requested here and looked at behind the tile's own loads.  One value alone is neither sought among eight nor
    // reduced over the wave ([512, 4096] 6.7 -> 6.4 us, [2048, 4096] 8.6 -> 8.2; read in front of the tile's loads 6.2 and 8.0).
    uint32_t part[TENSOR ? AMAX_MAX_WG / 64 : 1];
    if (TENSOR) {
#pragma unroll
        for (int u = 0; u < AMAX_MAX_WG / 64; ++u) part[u] = 0;
        part[0] = ((const uint32_t*)a.tensor_amax)[l < a.amax_parts ? l : 0];
        if (a.amax_parts > 64) {
#pragma unroll
            for (int u = 1; u < AMAX_MAX_WG / 64; ++u) part[u] = ((const uint32_t*)a.tensor_amax)[u * 64 + l < a.amax_parts ? u * 64 + l : 0];
        }
    }
    int pt, ct;
    if (!quant_tile_of_workgroup(a, block, pt, ct)) return;   // uniform over the workgroup
    const int64_t col0 = (int64_t)ct * QT;

    // ---- which source rows does this tile hold? ----
    int64_t src_row0 = 0;
    int rows_valid = 0;
    int64_t batch_off_rows = 0;  // TWOD: first row of this matrix in the flattened input
    int64_t out_row0;            // the tile's first row in the row-wise copy, and how many of its rows that has
    int rows_out;
    // K-step-major scales of a grouped transposed copy: the 16-byte scale panels restart at every group
    int64_t seg_pan0 = 0;        // panels of the groups in front of this tile's group
    int seg_tile = -1;           // this tile's number inside its group's padded segment (-1: not grouped)
    if (TWOD) {
        // grid.x enumerates (matrix, row tile); matrices are independent.
        const int tiles_per_mat = (int)((a.mat_rows + QT - 1) / QT);
        const int mat = pt / tiles_per_mat, rt = pt % tiles_per_mat;
        batch_off_rows = (int64_t)mat * a.mat_rows;
        src_row0 = batch_off_rows + (int64_t)rt * QT;
        int64_t rem = a.mat_rows - (int64_t)rt * QT;
        rows_valid = rem < QT ? (int)rem : QT;
        rem = a.out_rows - (int64_t)rt * QT;
        rows_out = rem < QT ? (int)rem : QT;
        out_row0 = (int64_t)mat * a.out_rows + (int64_t)rt * QT;
    } else if (!COL || a.group_lens == nullptr) {
        src_row0 = (int64_t)pt * QT;
        int64_t rem = a.rows - src_row0;
        rows_valid = rem <= 0 ? 0 : (rem < QT ? (int)rem : QT);
    } else {
        // every wave looks the tile's group up for itself
        GroupScan<> scan(a.rows, a.num_groups, l);
        uint32_t tiles = 0, pans = 0;
        for (int c = 0; c < a.num_groups; c += 64) {
            uint32_t first, end;
            scan.step(a.group_lens, c, first, end);
            const uint32_t nt = (end - first + QT - 1) / QT, np = (nt + 3) / 4;
            const uint32_t te = wave_prefix(nt) + tiles, pe = wave_prefix(np) + pans;
            const uint64_t hit = __ballot((uint32_t)pt >= te - nt && (uint32_t)pt < te);
            if (hit) {
                const int src = __builtin_ctzll(hit);
                seg_tile = pt - __builtin_amdgcn_readlane((int)(te - nt), src);
                seg_pan0 = (uint32_t)__builtin_amdgcn_readlane((int)(pe - np), src);
                const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)(end - first), src), r = (uint32_t)seg_tile * QT;
                src_row0 = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)first, src) + r;
                rows_valid = len - r < QT ? (int)(len - r) : QT;
                break;
            }
            tiles = (uint32_t)__builtin_amdgcn_readlane((int)te, 63);
            pans = (uint32_t)__builtin_amdgcn_readlane((int)pe, 63);
        }
        if (seg_tile < 0) {   // a padding tile behind the last group: its scales go behind the last group's panels
            seg_pan0 = pans;
            seg_tile = pt - (int)tiles;
        }
    }
    if (!TWOD) out_row0 = src_row0, rows_out = rows_valid;

    // fused activation: the tile's 128 probabilities (and row-mask bits) are fetched once by 128 lanes and
    // handed round through LDS; fetched per lane and row they would double the number of load instructions
    __shared__ float prob_tile[ACT >= 0 ? QT : 1];
    __shared__ uint8_t live_tile[ACT >= 0 ? QT : 1];
    float my_rstd = 0.f;
    if (ACT == PRO_RMSNORM) {
        // only requested here; it is handed round after the tile's own loads have gone out
        if (t < QT && t < rows_valid) my_rstd = ((const float*)a.probs)[src_row0 + t];
    } else if (ACT >= 0) {
        if (t < QT) {
            const bool live = t < rows_valid && (a.row_mask == nullptr || a.row_mask[src_row0 + t] != 0);
            live_tile[t] = live ? 1 : 0;
            prob_tile[t] = live ? load_prob(a.probs, a.probs_bf16, src_row0 + t) : 0.f;
        }
        __syncthreads();
    }

    const int64_t col = col0 + 8 * c16;
    const bool col_ok = col < a.cols;      // source column exists
    const bool out_ok = col < a.row_ld;    // row-wise output column exists (padding is written as zeros)

    // ---- load 8 rows x 8 columns per lane ----
    uint4 d[8];
    uint4 norm_wv = make_uint4(0, 0, 0, 0);
    if (ACT == PRO_RMSNORM && col_ok) norm_wv = *(const uint4*)(a.norm_w + col);
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const int r = 32 * w + 8 * rg + it;
        d[it] = make_uint4(0, 0, 0, 0);
        if (col_ok && r < rows_valid) {
            if (ACT < 0) {
                d[it] = load16_streaming(a.x + (src_row0 + r) * a.cols + col);
            } else if (ACT == PRO_RMSNORM) {
                d[it] = load16_streaming(a.x + (src_row0 + r) * a.cols + col);
            } else {
                if (live_tile[r]) {
                    const uint16_t* xr = a.x + (src_row0 + r) * 2 * a.cols + col;
                    d[it] = glu8<(ACT == MXL_ACT_GELU ? MXL_ACT_GELU : MXL_ACT_SILU)>(load16_streaming(xr),
                                                                                      load16_streaming(xr + a.cols),
                                                                                      prob_tile[r]);
                }
            }
        }
    }

    float tscale = 1.f;
    bool tensor_bad = false;   // abs-max is NaN or Inf: every code becomes NaN
    if (TENSOR) {
        // bit patterns of non-negative floats order like integers, a NaN above every number
        uint32_t bits = part[0];
        if (a.amax_parts > 1) {
#pragma unroll
            for (int u = 1; u < AMAX_MAX_WG / 64; ++u) bits = max(bits, part[u]);
#pragma unroll
            for (int s = 32; s > 0; s >>= 1) bits = max(bits, (uint32_t)__shfl_xor((int)bits, s));
        }
        bits = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits);
        const float amax = __uint_as_float(bits);
        tensor_bad = !(amax < __uint_as_float(0x7F800000u));
        tscale = (FMT == kFmtE5M2 ? 57344.f : 448.f) / fmaxf(amax, 1e-12f);
        if (block == 0 && t == 0 && a.scale_inv_out) *a.scale_inv_out = 1.0f / tscale;     // (workgroup 0 always has a tile)
    }

    if (ACT == PRO_RMSNORM) {
        if (t < QT) prob_tile[t] = my_rstd;
        __syncthreads();
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int r = 32 * w + 8 * rg + it;
            if (col_ok && r < rows_valid) d[it] = norm8(d[it], norm_wv, prob_tile[r]);
        }
    }

    // ---- block maxima ----
    uint32_t rmax[8];  // per row: max over the lane's 8 columns, then over the 32-column block
    uint32_t cmax[4] = {0, 0, 0, 0};  // per column pair (packed): max over the lane's 8 rows
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const uint32_t p0 = d[it].x & 0x7FFF7FFFu, p1 = d[it].y & 0x7FFF7FFFu, p2 = d[it].z & 0x7FFF7FFFu,
                       p3 = d[it].w & 0x7FFF7FFFu;
        if (COL && !TWOD && !RHT) {
            cmax[0] = pk_max16(cmax[0], p0);
            cmax[1] = pk_max16(cmax[1], p1);
            cmax[2] = pk_max16(cmax[2], p2);
            cmax[3] = pk_max16(cmax[3], p3);
        }
        uint32_t m = pk_max16(pk_max16(p0, p1), pk_max16(p2, p3));
        m = hmax16(m);
        m = max(m, dpp_xor1(m));
        m = max(m, dpp_xor2(m));
        rmax[it] = m;
    }
    uint32_t tile_byte = 0;
    if (TWOD) {
        uint32_t m = rmax[0];
#pragma unroll
        for (int it = 1; it < 8; ++it) m = max(m, rmax[it]);
        m = max(m, (uint32_t)__shfl_xor((int)m, 16));
        m = max(m, (uint32_t)__shfl_xor((int)m, 32));
        tile_byte = block_byte<FMT, SMODE>(m);
        // the transposed copy's scales without its codes: the tile's byte for each of the lane's 8 columns
        if (!COL && a.s_colT != nullptr && rg == 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) ((uint8_t*)scol_tile)[(8 * c16 + j) * 4 + w] = (uint8_t)tile_byte;
        }
    } else if (COL && !RHT) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cmax[j] = pk_max16(cmax[j], (uint32_t)__shfl_xor((int)cmax[j], 16));
            cmax[j] = pk_max16(cmax[j], (uint32_t)__shfl_xor((int)cmax[j], 32));
        }
    }

    // ---- row-wise copy ----
    if (ROW) {
        // (products of 64 bits once per lane: a multiplication costs four other instructions)
        const uint64_t sr_row = SR ? (uint64_t)(src_row0 + 32 * w + 8 * rg) * (uint64_t)(a.cols >> 1) + (uint64_t)(col >> 1) : 0;
        uint2 o_even = make_uint2(0u, 0u);   // FP8: codes of the even row of a row pair, kept until its partner is done
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int r = 32 * w + 8 * rg + it;
            const uint32_t byte = TWOD ? tile_byte : block_byte<FMT, SMODE>(rmax[it]);
            if ((c16 & 3) == 0) ((uint8_t*)srow_tile)[r * 4 + (c16 >> 2)] = (uint8_t)byte;
            if (!FP4) {
                uint2 o;
                if (TENSOR) {
                    o.x = tensor_bad ? 0x7F7F7F7Fu : cvt4_fp8<FMT>(d[it].x, d[it].y, tscale);
                    o.y = tensor_bad ? 0x7F7F7F7Fu : cvt4_fp8<FMT>(d[it].z, d[it].w, tscale);
                } else if (byte != 255u) {
                    const float inv = inv_scale(byte);
                    o.x = cvt4_e4m3(d[it].x, d[it].y, inv);
                    o.y = cvt4_e4m3(d[it].z, d[it].w, inv);
                } else {
                    o.x = nonfinite4_e4m3(d[it].x, d[it].y);
                    o.y = nonfinite4_e4m3(d[it].z, d[it].w);
                }
                // Two rows at a time, 16 bytes per lane: a lane pair swaps one 8-byte piece, after which the even lane
                // holds 16 consecutive codes of the even row and the odd lane 16 of the odd row.  Half the store
                // instructions, and in the K-step-major layout (64-byte row pieces, two rows to a cache line) an
                // instruction then writes whole lines.
                if ((it & 1) == 0) {
                    o_even = o;
                } else {
                    const bool odd = (c16 & 1) != 0;
                    const uint2 send = odd ? o_even : o;
                    const uint2 recv = make_uint2(dpp_xor1(send.x), dpp_xor1(send.y));
                    const uint4 out = odd ? make_uint4(recv.x, recv.y, o.x, o.y) : make_uint4(o_even.x, o_even.y, recv.x, recv.y);
                    const int rr = odd ? r : r - 1;
                    const int cc = c16 & ~1;          // the pair's first 8-column piece
                    if (out_ok && rr < rows_out) {
                        const int64_t at = a.kchunk == 2 ? ((int64_t)(2 * ct + (cc >> 3)) * a.chunk_rows_row + out_row0 + rr) * (QT / 2) + 8 * (cc & 7)
                                         : a.kchunk  ? ((int64_t)ct * a.chunk_rows_row + out_row0 + rr) * QT + 8 * cc
                                                     : (out_row0 + rr) * a.row_ld + col0 + 8 * cc;
                        store16(a.q_row + at, out, a.keep_row);
                    }
                }
            } else {
                uint32_t o;
                if (SR && byte != 255u) {
                    const float inv = inv_scale(byte);
                    const uint64_t key = sr_row + (uint64_t)it * (uint64_t)(a.cols >> 1);
                    o = sr8_e2m1(d[it].x, d[it].y, d[it].z, d[it].w, inv, key, a.sr_seed, 0);
                } else if (byte != 255u) {
                    const float sc = fwd_scale(byte);
                    o = cvt2_e2m1(d[it].x, sc) | (cvt2_e2m1(d[it].y, sc) << 8) | (cvt2_e2m1(d[it].z, sc) << 16) |
                        (cvt2_e2m1(d[it].w, sc) << 24);
                } else {
                    o = nonfinite2_e2m1(d[it].x) | (nonfinite2_e2m1(d[it].y) << 8) | (nonfinite2_e2m1(d[it].z) << 16) |
                        (nonfinite2_e2m1(d[it].w) << 24);
                }
                if (out_ok && r < rows_out) {
                    // element offsets; K-step-major: 64 elements (32 bytes) of a row per K step
                    const int64_t at = a.kchunk == 2 ? ((int64_t)(2 * ct + (c16 >> 3)) * a.chunk_rows_row + out_row0 + r) * (QT / 2) + 8 * (c16 & 7)
                                     : a.kchunk ? ((int64_t)ct * a.chunk_rows_row + out_row0 + r) * QT + 8 * c16
                                                : (out_row0 + r) * a.row_ld + col;
                    store4(a.q_row + at / 2, o, a.keep_row);
                }
            }
        }
    }

    // ---- Hadamard transform along the rows, in place (the row-wise copy above used the plain input) ----
    if (RHT) {
        // a 16-row group = the 8 rows of this lane and the 8 rows of the lane 16 further (rg ^ 1)
        const uint32_t upper = rg & 1;
        uint32_t* tw = (uint32_t*)d;
#pragma unroll
        for (int j2 = 0; j2 < 4; ++j2) {
            float lo[8], hi[8];
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const uint32_t flip = ((a.rht_signs >> (8 * upper + it)) & 1u) ? 0x80008000u : 0u;
                const uint32_t v = tw[it * 4 + j2] ^ flip;
                lo[it] = bf16_lo(v);
                hi[it] = bf16_hi(v);
            }
#pragma unroll
            for (int st = 1; st < 8; st <<= 1) {
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    if (it & st) continue;
                    const float a0 = lo[it], b0 = lo[it + st], a1 = hi[it], b1 = hi[it + st];
                    lo[it] = a0 + b0;
                    lo[it + st] = a0 - b0;
                    hi[it] = a1 + b1;
                    hi[it + st] = a1 - b1;
                }
            }
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const float o0 = __shfl_xor(lo[it], 16), o1 = __shfl_xor(hi[it], 16);
                const float r0 = upper ? (o0 - lo[it]) : (lo[it] + o0);
                const float r1 = upper ? (o1 - hi[it]) : (hi[it] + o1);
                tw[it * 4 + j2] = pack_bf16(r0 * 0.25f, r1 * 0.25f);
            }
        }
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            cmax[0] = pk_max16(cmax[0], d[it].x & 0x7FFF7FFFu);
            cmax[1] = pk_max16(cmax[1], d[it].y & 0x7FFF7FFFu);
            cmax[2] = pk_max16(cmax[2], d[it].z & 0x7FFF7FFFu);
            cmax[3] = pk_max16(cmax[3], d[it].w & 0x7FFF7FFFu);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cmax[j] = pk_max16(cmax[j], (uint32_t)__shfl_xor((int)cmax[j], 16));
            cmax[j] = pk_max16(cmax[j], (uint32_t)__shfl_xor((int)cmax[j], 32));
        }
    }

    // ---- column-wise (transposed) copy into the LDS tile ----
    if (COL) {
        // position of the lane's 8 rows along the padded token axis, in its first column
        const uint64_t sr_col = SR ? (uint64_t)col * (uint64_t)(a.W >> 1) + (((uint64_t)pt * QT + (uint64_t)(32 * w + 8 * rg)) >> 1) : 0;
        const uint32_t* dw = (const uint32_t*)d;  // dw[it*4 + j]: columns 2j, 2j+1 of row `it`
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t amax = (j & 1) ? (cmax[j >> 1] >> 16) : (cmax[j >> 1] & 0xFFFFu);
            const uint32_t byte = TWOD ? tile_byte : block_byte<FMT, SMODE>(amax);
            const int c = 8 * c16 + j;
            if (rg == 0) ((uint8_t*)scol_tile)[c * 4 + w] = (uint8_t)byte;
            // the lane's 8 rows of column j, as 4 packed (row 2i, row 2i+1) pairs
            uint32_t pr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t lo = dw[(2 * i) * 4 + (j >> 1)], hi = dw[(2 * i + 1) * 4 + (j >> 1)];
                pr[i] = (j & 1) ? ((lo >> 16) | (hi & 0xFFFF0000u)) : ((lo & 0xFFFFu) | (hi << 16));
            }
            if (!FP4) {
                uint2 o;
                if (TENSOR) {
                    o.x = tensor_bad ? 0x7F7F7F7Fu : cvt4_fp8<FMT>(pr[0], pr[1], tscale);
                    o.y = tensor_bad ? 0x7F7F7F7Fu : cvt4_fp8<FMT>(pr[2], pr[3], tscale);
                } else if (byte != 255u) {
                    const float inv = inv_scale(byte);
                    o.x = cvt4_e4m3(pr[0], pr[1], inv);
                    o.y = cvt4_e4m3(pr[2], pr[3], inv);
                } else {
                    o.x = nonfinite4_e4m3(pr[0], pr[1]);
                    o.y = nonfinite4_e4m3(pr[2], pr[3]);
                }
                *(uint2*)(t_tile + c * TPITCH + 32 * w + 8 * rg) = o;
            } else {
                uint32_t o;
                if (SR && byte != 255u) {
                    const float inv = inv_scale(byte);
                    const uint64_t key = sr_col + (uint64_t)j * (uint64_t)(a.W >> 1);
                    o = sr8_e2m1(pr[0], pr[1], pr[2], pr[3], inv, key, a.sr_seed, 1);
                } else if (byte != 255u) {
                    const float sc = fwd_scale(byte);
                    o = cvt2_e2m1(pr[0], sc) | (cvt2_e2m1(pr[1], sc) << 8) | (cvt2_e2m1(pr[2], sc) << 16) |
                        (cvt2_e2m1(pr[3], sc) << 24);
                } else {
                    o = nonfinite2_e2m1(pr[0]) | (nonfinite2_e2m1(pr[1]) << 8) | (nonfinite2_e2m1(pr[2]) << 16) |
                        (nonfinite2_e2m1(pr[3]) << 24);
                }
                *(uint32_t*)(t_tile + c * TPITCH + (32 * w + 8 * rg) / 2) = o;
            }
        }
    }
    __syncthreads();

    // ---- scales: one dword (4 blocks) per row / per column of the tile ----
    if (ROW && t < QT && t < rows_out) {
        const int64_t sld = a.row_ld / 32;
        const int64_t nb = (a.row_ld - col0) / 32;  // valid blocks in this tile row
        uint8_t* dst = a.s_row + (out_row0 + t) * sld + col0 / 32;
        const uint32_t v = srow_tile[t];
        if (a.kchunk >= 2) {
            store_panel_scales(a.s_row + ((int64_t)(ct >> 2) * a.chunk_rows_row + out_row0 + t) * 16, ct & 3, v);
        } else if (nb >= 4 && (sld & 3) == 0) {
            *(uint32_t*)dst = v;
        } else {
            for (int b = 0; b < 4 && b < nb; ++b) dst[b] = (uint8_t)(v >> (8 * b));
        }
    }
    if (COL || (TWOD && a.s_colT != nullptr)) {
        const int64_t out_rows_base = TWOD ? (batch_off_rows / a.mat_rows) * a.cols : 0;  // TWOD: matrix * k
        const int64_t m0 = TWOD ? (src_row0 - batch_off_rows) : (int64_t)pt * QT;          // position along W
        if (t < QT && col0 + t < a.cols) {
            uint8_t* dst = a.s_colT + (out_rows_base + col0 + t) * (a.W / 32) + m0 / 32;
            const uint32_t v = scol_tile[t];
            const int64_t nb = (a.W - m0) / 32;
            if (a.kchunk >= 2) {
                const int64_t mt = seg_tile >= 0 ? (int64_t)seg_tile : m0 / QT;
                store_panel_scales(a.s_colT + ((seg_pan0 + mt / 4) * a.chunk_rows_col + out_rows_base + col0 + t) * 16, (int)(mt & 3), v);
            } else if (nb >= 4 && ((a.W / 32) & 3) == 0) {
                *(uint32_t*)dst = v;
            } else {
                for (int b = 0; b < 4 && b < nb; ++b) dst[b] = (uint8_t)(v >> (8 * b));
            }
        }
        if (!COL) return;                        // (scales only)
        constexpr int ROWB = FP4 ? QT / 2 : QT;  // bytes per transposed tile row
        constexpr int LPR = ROWB / 16;           // lanes per row
        const int64_t wbytes = FP4 ? a.W / 2 : a.W;
        const int64_t m0b = FP4 ? m0 / 2 : m0;
        const int64_t avail = wbytes - m0b;      // bytes left in the output row (TWOD tails)
#pragma unroll
        for (int i = 0; i < QT / (QTHREADS / LPR); ++i) {
            const int c = t / LPR + i * (QTHREADS / LPR);
            const int ch = t % LPR;
            if (col0 + c < a.cols && 16 * ch < avail) {
                const uint4 v = *(const uint4*)(t_tile + c * TPITCH + 16 * ch);
                const int64_t at = (FP4 && a.kchunk == 2)
                                       ? ((2 * (m0 / QT) + (ch >> 1)) * a.chunk_rows_col + out_rows_base + col0 + c) * (QT / 4) + 16 * (ch & 1)
                                   : a.kchunk == 2
                                       ? ((2 * (m0 / QT) + (ch >> 2)) * a.chunk_rows_col + out_rows_base + col0 + c) * (QT / 2) + 16 * (ch & 3)
                                   : a.kchunk ? ((m0 / QT) * a.chunk_rows_col + out_rows_base + col0 + c) * ROWB + 16 * ch
                                              : (out_rows_base + col0 + c) * wbytes + m0b + 16 * ch;
                store16(a.q_colT + at, v, a.keep_col);
            }
        }
    }
}

template <int FMT, int SMODE, bool ROW, bool COL, bool TWOD, int ACT = -1, bool SR = false, bool RHT = false>
__global__ __launch_bounds__(QTHREADS) void mx_quant_kernel(QuantArgs a) {
    quant_workgroup<FMT, SMODE, ROW, COL, TWOD, ACT, SR, RHT>(a, (int)blockIdx.x);
}

// The row-wise copy alone of few rows, K-step-major: a wave takes two rows of a 512-element scale panel, a lane 8 columns of both.
// A 128 x 128 tile's workgroup has four times the rows to a lane, one after the other, two barriers and a search for its tile, and
// few rows are few workgroups: what such a launch lasts is that chain.  Linear on cached weights, us on tiles / so: 64 rows of 4096 to 14336
// columns (as a graph, the host takes 18) 17.0 / 15.2, 256 rows 22.0 / 20.2, 512 33.1 / 31.9, [1024, 4096] x 4096 23.5 / 22.8, [2048, 4096] x
// 4096 39.8 / 38.8; E2M1, [512, 4096] x 14336 23.1 / 20.9, [1024, 4096] x 4096 18.9 / 17.5.  With more waves than the chip holds at once
// (32 to a CU: 8192) tiles are ahead, for narrow rows, whose waves are part empty, as for wide ones: quantiser alone, time so / on tiles, at
// 6144 waves 0.88 (3072 rows of 2048) to 0.97 (12288 of 128), at 8192 1.01 to 1.08, 65536 rows of 128 columns 1.49.  An RMSNorm in front
// moves the line up (8192 waves 0.90 to 1.00, 16384 1.15), a gated activation, which is what a tile's lane spends its time on, past the
// sizes here: 0.84 at 32768 rows of 256, 0.74 at 8192 of 1024.
constexpr int64_t FEW_ROWS_ELEMENTS = (int64_t)8 << 20;
static bool few_rows(const QuantArgs& a, int act) {
    if (a.rows * a.row_ld > FEW_ROWS_ELEMENTS) return false;      // (at most 65536 rows: 32768 pairs of them)
    const int64_t waves = (a.rows + 1) / 2 * ((a.row_ld + 511) / 512);
    return act == PRO_RMSNORM ? waves <= 8192 : act >= 0 || waves <= 6144;
}
template <int FMT, int SMODE, int ACT>
__global__ __launch_bounds__(64) void mx_quant_few_rows_kernel(QuantArgs a) {
    constexpr bool FP4 = (FMT == kFmtE2M1);
    const int l = threadIdx.x;
    const int64_t row0 = 2 * (int64_t)blockIdx.y, col = 512 * (int64_t)blockIdx.x + 8 * l;
    const bool two = row0 + 1 < a.rows;
    if (col >= a.row_ld) return;          // (row_ld is a multiple of 128: the 16 lanes of a K step stay or go together)
    uint4 d[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
    if (col < a.cols) {
        if (ACT < 0 || ACT == PRO_RMSNORM) {
            const uint16_t* x = a.x + row0 * a.cols + col;
            d[0] = load16_streaming(x);
            if (two) d[1] = load16_streaming(x + a.cols);
        }
        if (ACT == PRO_RMSNORM) {
            const uint4 wv = *(const uint4*)(a.norm_w + col);
            const float* rstd = (const float*)a.probs + row0;
            d[0] = norm8(d[0], wv, rstd[0]);
            if (two) d[1] = norm8(d[1], wv, rstd[1]);
        } else if (ACT >= 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if ((i == 0 || two) && (a.row_mask == nullptr || a.row_mask[row0 + i] != 0)) {
                    const uint16_t* x = a.x + (row0 + i) * 2 * a.cols + col;
                    d[i] = glu8<(ACT == MXL_ACT_GELU ? MXL_ACT_GELU : MXL_ACT_SILU)>(load16_streaming(x), load16_streaming(x + a.cols),
                                                                                      load_prob(a.probs, a.probs_bf16, row0 + i));
                }
            }
        }
    }
    uint32_t byte[2];
    uint2 o[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t m = hmax16(pk_max16(pk_max16(d[i].x & 0x7FFF7FFFu, d[i].y & 0x7FFF7FFFu), pk_max16(d[i].z & 0x7FFF7FFFu, d[i].w & 0x7FFF7FFFu)));
        m = max(m, dpp_xor1(m));
        m = max(m, dpp_xor2(m));
        byte[i] = scale_byte<FMT, SMODE>(m);
        if (FP4) {
            const float sc = fwd_scale(byte[i]);
            o[i].x = byte[i] != 255u ? cvt2_e2m1(d[i].x, sc) | (cvt2_e2m1(d[i].y, sc) << 8) | (cvt2_e2m1(d[i].z, sc) << 16) | (cvt2_e2m1(d[i].w, sc) << 24)
                                     : nonfinite2_e2m1(d[i].x) | (nonfinite2_e2m1(d[i].y) << 8) | (nonfinite2_e2m1(d[i].z) << 16) |
                                           (nonfinite2_e2m1(d[i].w) << 24);
        } else if (byte[i] != 255u) {
            const float inv = inv_scale(byte[i]);
            o[i] = make_uint2(cvt4_e4m3(d[i].x, d[i].y, inv), cvt4_e4m3(d[i].z, d[i].w, inv));
        } else {
            o[i] = make_uint2(nonfinite4_e4m3(d[i].x, d[i].y), nonfinite4_e4m3(d[i].z, d[i].w));
        }
    }
    const int64_t step = FP4 ? col >> 7 : col >> 6;                  // 64 bytes of a row either way
    uint8_t* q = a.q_row + (step * a.chunk_rows_row + row0) * 64;
    if (FP4) {
        store4(q + 4 * (l & 15), o[0].x, a.keep_row);
        if (two) store4(q + 64 + 4 * (l & 15), o[1].x, a.keep_row);
    } else {
        // a lane pair swaps 8-byte pieces: the even lane 16 codes of the first row, the odd lane 16 of the second
        const bool odd = (l & 1) != 0;
        const uint2 send = odd ? o[0] : o[1];
        const uint2 recv = make_uint2(dpp_xor1(send.x), dpp_xor1(send.y));
        if (!odd || two)
            store16(q + (odd ? 64 : 0) + 8 * (l & 6), odd ? make_uint4(recv.x, recv.y, o[1].x, o[1].y) : make_uint4(o[0].x, o[0].y, recv.x, recv.y), a.keep_row);
    }
    // block b = l / 4 of the panel at [block parity][K step]; the second lane of a block writes the second row's byte
    const int sub = l & 3, b = l >> 2;
    if (sub == 0 || (sub == 1 && two))
        a.s_row[((int64_t)blockIdx.x * a.chunk_rows_row + row0 + sub) * 16 + 8 * (b & 1) + (b >> 1)] = (uint8_t)(sub ? byte[1] : byte[0]);
}

// Both operands of a linear's forward in one launch: the activations' two copies (the first x_wgs workgroups) and the
// weight's (WCOL: its transposed codes too).  Neither fills the chip for long where the linear is small, and each launch
// costs its fill and drain and the gap behind it.  Forward of a linear, quantisers and GEMM, two launches / one, us:
// [256, 4096] x 4096 39.8 / 34.0; [1999, 2880] x 5760 67.9 / 62.8; [8192, 4096] x 14336 422 / 412; tensor-wise [4096, 14336] x
// 4096 279 / 272; 8 experts of [2048, 2048], 2048 rows, 56 / 51.  The weight's workgroups hold the activations' 108 registers
// a lane instead of 58, 4 waves per SIMD instead of 8, and large experts are mostly weight: 32 x [4096, 7168], 8192 rows, 860 /
// 865; 8 x [28672, 4096], 512 rows, 694 / 668.  The input may be transformed by Hadamard, or formed by an RMSNorm from
// statistics that are there already.
template <int FMT, int SMODE, bool WCOL, int ACT = -1, bool RHT = false>
__global__ __launch_bounds__(QTHREADS) void mx_quant_pair_kernel(QuantArgs x, QuantArgs w, unsigned x_wgs) {
    if (blockIdx.x < x_wgs) quant_workgroup<FMT, SMODE, true, true, false, ACT, false, RHT>(x, (int)blockIdx.x);
    else quant_workgroup<FMT, SMODE, true, WCOL, true>(w, (int)(blockIdx.x - x_wgs));
}

// ---------------------------------------------------------------------------
// dequantise: codes + scales -> bf16 (row-wise layout)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float dec_e4m3(uint32_t c) {
    // exact decode through fp32 bit assembly
    const uint32_t s = (c & 0x80u) << 24, e = (c >> 3) & 0xFu, m = c & 7u;
    float v;
    if (e == 0)
        v = (float)m * 0.001953125f;  // m * 2^-9
    else if ((c & 0x7Fu) == 0x7Fu)
        v = __uint_as_float(0x7FC00000u);
    else
        v = __uint_as_float(((e + 120u) << 23) | (m << 20));
    return __uint_as_float(__float_as_uint(v) | s);
}
// E5M2 is the upper byte of an IEEE half: exact through the half -> float conversion (NaN and infinity included)
__device__ __forceinline__ float dec_e5m2(uint32_t c) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(c << 8));
}
__device__ __forceinline__ float dec_e2m1(uint32_t c) {
    const uint32_t s = (c & 8u) << 28, e = (c >> 1) & 3u, m = c & 1u;
    const uint32_t bits = e ? (((e + 126u) << 23) | (m << 22)) : (m ? 0x3F000000u : 0u);
    return __uint_as_float(bits | s);
}

template <int FMT>
__global__ __launch_bounds__(256) void mx_dequant_kernel(const uint8_t* q, const uint8_t* s, uint16_t* out,
                                                         int64_t nblocks) {
    // one lane per 8 elements; 4 lanes per MX block
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t blk = i >> 2;
    if (blk >= nblocks) return;
    const uint32_t byte = s[blk];
    // fp32 holds 2^(byte-127) exactly (subnormal for byte 0); multiply in two steps to stay exact
    const float sc = (byte == 255u) ? __uint_as_float(0x7FC00000u) : fwd_scale(byte);
    float v[8];
    if (FMT == kFmtE4M3 || FMT == kFmtE5M2) {
        const uint2 c = *(const uint2*)(q + i * 8);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = FMT == kFmtE5M2 ? dec_e5m2((c.x >> (8 * k)) & 0xFFu) : dec_e4m3((c.x >> (8 * k)) & 0xFFu);
            v[4 + k] = FMT == kFmtE5M2 ? dec_e5m2((c.y >> (8 * k)) & 0xFFu) : dec_e4m3((c.y >> (8 * k)) & 0xFFu);
        }
    } else {
        const uint32_t c = *(const uint32_t*)(q + i * 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = dec_e2m1((c >> (4 * k)) & 0xFu);
    }
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v2bf h = {(__bf16)(v[2 * k] * sc), (__bf16)(v[2 * k + 1] * sc)};
        o[k] = __builtin_bit_cast(uint32_t, h);
    }
    *(uint4*)(out + i * 8) = make_uint4(o[0], o[1], o[2], o[3]);
}

// ---------------------------------------------------------------------------
// host-side dispatch
// ---------------------------------------------------------------------------
// the activations of a pair, prepared and not yet launched; lives on the stack of the call that launches both
struct HeldQuant {
    bool held = false;
    int fmt, smode;          // smode: SCALE_TENSOR or an MXL_SCALE_*
    int act;                 // -1 or PRO_RMSNORM
    bool rht;
    QuantArgs a;
    int64_t wgs;
};

// `keep`: the caller's word that codes stored through the caches are found there by the GEMM behind (mx_linear.hip: keeps), for
// copies that fit the 256 MiB memory-side cache; the transposed ones are read later, the activations' not before the backward,
// and may take a quarter of it.
constexpr int64_t KEEP_ROW_BYTES = (int64_t)256 << 20, KEEP_COL_BYTES = KEEP_ROW_BYTES / 4;
static void keep_in_cache(QuantArgs& a, bool keep, int fmt, int64_t row_codes, int64_t col_codes) {
    const int per = fmt == MXL_FMT_E2M1 ? 2 : 1;
    a.keep_row = keep && row_codes / per <= KEEP_ROW_BYTES;
    a.keep_col = keep && col_codes / per <= KEEP_COL_BYTES;
}

// fills in the launch's tile grid; its workgroups
static int quant_grid(QuantArgs& a, int64_t tiles_r, int64_t tiles_c, int64_t* wgs) {
    const int lg = a.kchunk >= 2 ? 2 : 3;
    const int64_t side = (int64_t)1 << lg, super_r = (tiles_r + side - 1) / side, super_c = (tiles_c + side - 1) / side;
    const int64_t n_super = super_r * super_c;
    *wgs = (n_super + 7) / 8 * 8 * side * side;
    if (tiles_r > 0x7FFFFFFF || tiles_c > 0x7FFFFFFF || *wgs > 0x7FFFFFFF) return MXL_EINVAL;
    if (!device_is_gfx950()) return MXL_ENODEV;
    a.tiles_r = (int)tiles_r;
    a.tiles_c = (int)tiles_c;
    a.super_c = (int)super_c;
    a.super_log = lg;
    a.n_super = (int)n_super;
    return MXL_OK;
}

template <int FMT, int SMODE, bool TWOD, int ACT = -1, bool SR = false, bool RHT = false>
static int launch_quant(QuantArgs& a, int64_t tiles_r, int64_t tiles_c, hipStream_t st) {
    int64_t wgs;
    if (const int rc = quant_grid(a, tiles_r, tiles_c, &wgs)) return rc;
    const dim3 grid((unsigned)wgs);
    const bool row = a.q_row != nullptr, col = a.q_colT != nullptr;
    if constexpr (FMT != MXL_FMT_E5M2 && SMODE != SCALE_TENSOR && !TWOD && !SR && !RHT) {
        if (row && !col && a.kchunk >= 2 && few_rows(a, ACT)) {
            const dim3 pairs((unsigned)((a.row_ld + 511) / 512), (unsigned)((a.rows + 1) / 2));
            hipLaunchKernelGGL((mx_quant_few_rows_kernel<FMT, SMODE, ACT>), pairs, dim3(64), 0, st, a);
            return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
        }
    }
    if (row && col)
        hipLaunchKernelGGL((mx_quant_kernel<FMT, SMODE, true, true, TWOD, ACT, SR, RHT>), grid, dim3(QTHREADS), 0, st, a);
    else if (row && !RHT)
        hipLaunchKernelGGL((mx_quant_kernel<FMT, SMODE, true, false, TWOD, ACT, SR, false>), grid, dim3(QTHREADS), 0, st,
                           a);
    else if (ACT < 0 && col)
        hipLaunchKernelGGL((mx_quant_kernel<FMT, SMODE, false, true, TWOD, -1, SR, RHT>), grid, dim3(QTHREADS), 0, st, a);
    else
        return MXL_EINVAL;   // the fused activation always feeds a forward GEMM: a row-wise copy is part of it
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

template <bool TWOD, int ACT = -1>
static int dispatch_quant(int fmt, int smode, QuantArgs& a, int64_t tiles_r, int64_t tiles_c, hipStream_t st) {
#define MXL_Q(F, S) \
    if (fmt == F && smode == S) return launch_quant<F, S, TWOD, ACT>(a, tiles_r, tiles_c, st);
    MXL_Q(MXL_FMT_E4M3, MXL_SCALE_OCP_FLOOR)
    MXL_Q(MXL_FMT_E4M3, MXL_SCALE_RCEIL)
    MXL_Q(MXL_FMT_E4M3, MXL_SCALE_EVEN)
    MXL_Q(MXL_FMT_E2M1, MXL_SCALE_OCP_FLOOR)
    MXL_Q(MXL_FMT_E2M1, MXL_SCALE_RCEIL)
    MXL_Q(MXL_FMT_E2M1, MXL_SCALE_EVEN)
#undef MXL_Q
    return MXL_EINVAL;
}

// the MXFP4 recipe's options (1-D E2M1 only): stochastic rounding, Hadamard transform of the transposed copy
template <bool SR, bool RHT>
static int dispatch_quant_fp4(int smode, QuantArgs& a, int64_t tiles_r, int64_t tiles_c, hipStream_t st) {
    if (smode == MXL_SCALE_OCP_FLOOR)
        return launch_quant<MXL_FMT_E2M1, MXL_SCALE_OCP_FLOOR, false, -1, SR, RHT>(a, tiles_r, tiles_c, st);
    if (smode == MXL_SCALE_RCEIL) return launch_quant<MXL_FMT_E2M1, MXL_SCALE_RCEIL, false, -1, SR, RHT>(a, tiles_r, tiles_c, st);
    if (smode == MXL_SCALE_EVEN) return launch_quant<MXL_FMT_E2M1, MXL_SCALE_EVEN, false, -1, SR, RHT>(a, tiles_r, tiles_c, st);
    return MXL_EINVAL;
}

// tensor-wise scaling: E4M3 or E5M2 codes, 1-D (activations, gradients) or batched-matrix (weights) tiling
template <bool TWOD>
static int dispatch_quant_tensor(int fmt, QuantArgs& a, int64_t tiles_r, int64_t tiles_c, hipStream_t st) {
    if (fmt == MXL_FMT_E4M3) return launch_quant<MXL_FMT_E4M3, SCALE_TENSOR, TWOD>(a, tiles_r, tiles_c, st);
    if (fmt == MXL_FMT_E5M2) return launch_quant<MXL_FMT_E5M2, SCALE_TENSOR, TWOD>(a, tiles_r, tiles_c, st);
    return MXL_EINVAL;
}

// the kernel for both quantisations of a pair; null: there is none, and each is launched by itself
typedef void (*QuantPairKernel)(QuantArgs, QuantArgs, unsigned);
static QuantPairKernel pair_kernel(const HeldQuant& x, int fmt, int smode, const QuantArgs& w) {
    if (x.fmt != fmt || x.smode != smode || !x.a.q_row || !x.a.q_colT || !w.q_row) return nullptr;
#define MXL_QP(F, S, ACT, RHT)                                              \
    if (fmt == F && smode == S && x.act == ACT && x.rht == RHT)             \
        return w.q_colT ? (QuantPairKernel)mx_quant_pair_kernel<F, S, true, ACT, RHT> : (QuantPairKernel)mx_quant_pair_kernel<F, S, false, ACT, RHT>;
    MXL_QP(MXL_FMT_E4M3, MXL_SCALE_OCP_FLOOR, -1, false)
    MXL_QP(MXL_FMT_E4M3, MXL_SCALE_OCP_FLOOR, PRO_RMSNORM, false)
    MXL_QP(MXL_FMT_E2M1, MXL_SCALE_OCP_FLOOR, -1, false)
    MXL_QP(MXL_FMT_E2M1, MXL_SCALE_OCP_FLOOR, -1, true)
    MXL_QP(MXL_FMT_E4M3, SCALE_TENSOR, -1, false)
#undef MXL_QP
    return nullptr;
}
static int launch_quant_pair(QuantPairKernel kern, const HeldQuant& x, QuantArgs& w, int64_t tiles_r, int64_t tiles_c, hipStream_t st) {
    int64_t wgs;
    if (const int rc = quant_grid(w, tiles_r, tiles_c, &wgs)) return rc;
    if (x.wgs + wgs > 0x7FFFFFFF) return MXL_EINVAL;
    hipLaunchKernelGGL(kern, dim3((unsigned)(x.wgs + wgs)), dim3(QTHREADS), 0, st, x.a, w, (unsigned)x.wgs);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

// abs-max of one or two bf16 tensors: non-negative floats order like their bit patterns, so an integer atomic max on
// the fp32 pattern does it (a NaN pattern is larger than every number and wins).  One atomic per workgroup.
//
// Bound by reading the tensor once, if enough loads are in flight and few enough atomics meet at the one result: a
// workgroup takes pieces of 32 KiB, eight 16-byte loads per lane issued together, and at most AMAX_MAX_WG of them share
// a tensor.  [4096, 14336] twice: 103 us with one load in flight per lane and up to 4096 workgroups, 41 (5.8 TB/s) so;
// [4096, 4096]: 17.4 -> 11.8 us (16.6 with 1024 workgroups).
// The loads are ordinary ones: the quantiser reads the same tensor next, and up to 256 MiB of it then come from the
// memory-side cache.
constexpr int AMAX_LOADS = 8, AMAX_PIECE = 256 * AMAX_LOADS;
struct AmaxArgs {
    const uint16_t* x[2];
    int64_t n[2];
    uint32_t* out[2];
    uint32_t wg[2];          // workgroups of each tensor
    int parts;               // every workgroup stores its own maximum, out[tensor][workgroup]; nothing is initialised
};
__global__ __launch_bounds__(256) void amax_kernel(AmaxArgs p) {
    __shared__ uint32_t part[4];
    const int second = blockIdx.x >= p.wg[0];
    const uint16_t* x = p.x[second];
    const int64_t n = p.n[second], n8 = n / 8, wg = p.wg[second];
    const int64_t blk = (int64_t)blockIdx.x - (second ? p.wg[0] : 0u);
    uint32_t m = 0;
    for (int64_t i0 = blk * AMAX_PIECE; i0 < n8; i0 += wg * AMAX_PIECE) {
        uint4 v[AMAX_LOADS];
#pragma unroll
        for (int u = 0; u < AMAX_LOADS; ++u) {
            // past the end: the last piece once more
            const int64_t i = i0 + u * 256 + threadIdx.x;
            v[u] = *(const uint4*)(x + (i < n8 ? i : n8 - 1) * 8);
        }
#pragma unroll
        for (int u = 0; u < AMAX_LOADS; ++u)
            m = pk_max16(m, pk_max16(pk_max16(v[u].x & 0x7FFF7FFFu, v[u].y & 0x7FFF7FFFu), pk_max16(v[u].z & 0x7FFF7FFFu, v[u].w & 0x7FFF7FFFu)));
    }
    m = hmax16(m);
    if (blk == 0 && threadIdx.x == 0)
        for (int64_t i = n8 * 8; i < n; ++i) m = max(m, (uint32_t)(x[i] & 0x7FFFu));   // tail of fewer than 8 elements
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, s));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(part[0], part[1]), max(part[2], part[3]));
        // bf16 pattern -> fp32 pattern
        if (p.parts) p.out[second][blk] = m << 16;
        else atomicMax(p.out[second], m << 16);
    }
}

__global__ void amax_init_kernel(uint32_t* a, uint32_t* b) {
    *a = 0u;
    *b = 0u;
}

static uint32_t amax_workgroups(int64_t n) {
    const int64_t pieces = (n / 8 + AMAX_PIECE - 1) / AMAX_PIECE;
    if (pieces <= 0) return n > 0 ? 1 : 0;
    const int64_t rounds = (pieces + AMAX_MAX_WG - 1) / AMAX_MAX_WG;
    return (uint32_t)((pieces + rounds - 1) / rounds);      // every workgroup the same number of pieces
}

int amax_parts(int64_t n) { return (int)amax_workgroups(n); }

// out_a = max |a| over na values, out_b = max |b| (b may be null: one tensor), in two launches; with `parts` the
// amax_parts(na) and amax_parts(nb) maxima of the workgroups, na and nb > 0, in one (the initialising launch costs a linear
// 5 us in each direction, more than the quantiser's look at 512 values)
int amax_pair(const void* a, int64_t na, void* out_a, const void* b, int64_t nb, void* out_b, bool parts, void* stream) {
    if (na < 0 || nb < 0 || !out_a || (na > 0 && !a) || ((uintptr_t)a & 15) != 0) return MXL_EINVAL;
    if (nb > 0 && (!b || !out_b || ((uintptr_t)b & 15) != 0)) return MXL_EINVAL;
    if (!device_is_gfx950()) return MXL_ENODEV;
    hipStream_t st = (hipStream_t)stream;
    AmaxArgs p{{(const uint16_t*)a, (const uint16_t*)b}, {na, nb}, {(uint32_t*)out_a, (uint32_t*)(out_b ? out_b : out_a)},
               {amax_workgroups(na), amax_workgroups(nb)}, parts};
    if (!parts) {
        // a fill kernel, not a memset: callers may be capturing the stream into a graph
        hipLaunchKernelGGL(amax_init_kernel, dim3(1), dim3(1), 0, st, p.out[0], p.out[1]);
        if (hipGetLastError() != hipSuccess) return MXL_ELAUNCH;
    }
    if (p.wg[0] + p.wg[1] == 0) return MXL_OK;
    hipLaunchKernelGGL(amax_kernel, dim3(p.wg[0] + p.wg[1]), dim3(256), 0, st, p);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

}  // namespace mxl

using namespace mxl;

extern "C" int mxl_amax(const void* x_bf16, int64_t n, void* amax_f32, void* stream) {
    return amax_pair(x_bf16, n, amax_f32, nullptr, 0, nullptr, false, stream);
}

extern "C" int64_t mxl_padded_width(int64_t total_rows, int num_groups) {
    if (num_groups < 1) num_groups = 1;
    return (total_rows + (int64_t)(MXL_SEG_ALIGN - 1) * num_groups) / MXL_SEG_ALIGN * MXL_SEG_ALIGN;
}

// code layout selected by the flags: 0 row-major, 1 K-chunk-major, 2 K-step-major, 3 K-step-major with steps of 128
// elements (E2M1 only: 64-byte rows, i.e. K-chunk-major codes with K-step-major scale panels), -1 contradictory flags
static int qf_layout(uint32_t flags) {
    if ((flags & MXL_QF_KCHUNK) && (flags & MXL_QF_KSTEP)) return -1;
    if ((flags & MXL_QF_KSTEP128) && !(flags & MXL_QF_KSTEP)) return -1;
    return (flags & MXL_QF_KSTEP128) ? 3 : (flags & MXL_QF_KSTEP) ? 2 : (flags & MXL_QF_KCHUNK) ? 1 : 0;
}

static int quantize_1d(const void* x_bf16, int64_t rows, int64_t cols, int64_t row_ld, int fmt, int scale_mode,
                       const int64_t* group_lens, int num_groups, void* q_row, void* s_row, void* q_colT, void* s_colT,
                       int act, const void* probs, int probs_dtype, const uint8_t* row_mask, void* stream,
                       bool sr = false, uint64_t sr_seed = 0, bool rht = false, uint32_t rht_signs = 0,
                       int kchunk = 0, const void* norm_w = nullptr, const void* tensor_amax = nullptr,
                       void* scale_inv_out = nullptr, HeldQuant* hold = nullptr, int parts = 1, bool keep = false) {
    if (row_ld == 0) row_ld = cols;
    if (kchunk < 0) return MXL_EINVAL;                  // contradictory layout flags
    if (kchunk == 2 && fmt == MXL_FMT_E2M1) kchunk = 3;  // E2M1 activations: the K step is 128 elements (64-byte rows)
    if (kchunk == 3 && fmt != MXL_FMT_E2M1) return MXL_EINVAL;
    if (kchunk && q_row && row_ld % QT != 0) return MXL_EINVAL;   // whole 128-element chunks
    if ((sr || rht) && (fmt != MXL_FMT_E2M1 || act >= 0)) return MXL_EINVAL;
    if (rht && !q_colT) return MXL_EINVAL;   // the transform belongs to the transposed copy
    if (row_ld < cols || row_ld % MXL_BLOCK != 0) return MXL_EINVAL;
    if ((!x_bf16 && rows > 0) || rows < 0 || cols <= 0 || cols % MXL_BLOCK != 0) return MXL_EINVAL;
    if ((q_row == nullptr) != (s_row == nullptr) || (q_colT == nullptr) != (s_colT == nullptr)) return MXL_EINVAL;
    if (!q_row && !q_colT) return MXL_EINVAL;
    if (num_groups < 0 || num_groups > MXL_MAX_GROUPS || (num_groups > 0) != (group_lens != nullptr)) return MXL_EINVAL;
    QuantArgs a;
    a.x = (const uint16_t*)x_bf16;
    a.rows = rows;
    a.cols = cols;
    a.group_lens = group_lens;
    a.num_groups = num_groups;
    a.q_row = (uint8_t*)q_row;
    a.s_row = (uint8_t*)s_row;
    a.q_colT = (uint8_t*)q_colT;
    a.s_colT = (uint8_t*)s_colT;
    a.row_ld = row_ld;
    a.W = mxl_padded_width(rows, num_groups);
    a.mat_rows = 0;
    a.out_rows = 0;
    a.probs = probs;
    a.probs_bf16 = probs_dtype == MXL_PROBS_BF16;
    a.row_mask = row_mask;
    a.norm_w = (const uint16_t*)norm_w;
    a.tensor_amax = (const float*)tensor_amax;
    a.amax_parts = parts;
    a.scale_inv_out = (float*)scale_inv_out;
    a.sr_seed = sr_seed;
    a.rht_signs = rht_signs & 0xFFFFu;
    a.kchunk = kchunk;
    a.chunk_rows_row = rows;
    a.chunk_rows_col = cols;
    keep_in_cache(a, keep, fmt, rows * row_ld, cols * a.W);
    const int64_t gx = q_colT ? a.W / QT : (rows + QT - 1) / QT;
    const int64_t gy = ((q_row ? row_ld : cols) + QT - 1) / QT;
    if (hold && gx > 0 && !sr && (act < 0 || act == PRO_RMSNORM)) {
        hold->held = true;
        hold->act = act;
        hold->rht = rht;
        hold->fmt = fmt;
        hold->smode = tensor_amax ? SCALE_TENSOR : scale_mode;
        hold->a = a;
        return quant_grid(hold->a, gx, gy, &hold->wgs);
    }
    if (tensor_amax) {
        if (sr || rht || act >= 0) return MXL_EINVAL;
        if (gx == 0) return MXL_OK;   // nothing to quantise (scale_inv_out is then left unwritten)
        return dispatch_quant_tensor<false>(fmt, a, gx, gy, (hipStream_t)stream);
    }
    if (gx == 0) return MXL_OK;
    if (sr && rht) return dispatch_quant_fp4<true, true>(scale_mode, a, gx, gy, (hipStream_t)stream);
    if (sr) return dispatch_quant_fp4<true, false>(scale_mode, a, gx, gy, (hipStream_t)stream);
    if (rht) return dispatch_quant_fp4<false, true>(scale_mode, a, gx, gy, (hipStream_t)stream);
    if (act == MXL_ACT_SILU) return dispatch_quant<false, MXL_ACT_SILU>(fmt, scale_mode, a, gx, gy, (hipStream_t)stream);
    if (act == MXL_ACT_GELU) return dispatch_quant<false, MXL_ACT_GELU>(fmt, scale_mode, a, gx, gy, (hipStream_t)stream);
    if (act == PRO_RMSNORM) return dispatch_quant<false, PRO_RMSNORM>(fmt, scale_mode, a, gx, gy, (hipStream_t)stream);
    return dispatch_quant<false>(fmt, scale_mode, a, gx, gy, (hipStream_t)stream);
}

extern "C" int mxl_quantize(const void* x_bf16, int64_t rows, int64_t cols, int64_t row_ld, int fmt, int scale_mode,
                            const int64_t* group_lens, int num_groups, void* q_row, void* s_row, void* q_colT,
                            void* s_colT, void* stream) {
    return quantize_1d(x_bf16, rows, cols, row_ld, fmt, scale_mode, group_lens, num_groups, q_row, s_row, q_colT, s_colT,
                       -1, nullptr, MXL_PROBS_F32, nullptr, stream);
}

extern "C" int mxl_quantize_ex(const void* x_bf16, int64_t rows, int64_t cols, int64_t row_ld, int fmt, int scale_mode,
                               const int64_t* group_lens, int num_groups, void* q_row, void* s_row, void* q_colT,
                               void* s_colT, uint32_t flags, uint64_t sr_seed, uint32_t rht_signs, void* stream) {
    if (flags & ~(uint32_t)(MXL_QF_SR | MXL_QF_RHT_COL | MXL_QF_KCHUNK | MXL_QF_KSTEP | MXL_QF_KSTEP128)) return MXL_EINVAL;
    return quantize_1d(x_bf16, rows, cols, row_ld, fmt, scale_mode, group_lens, num_groups, q_row, s_row, q_colT,
                       s_colT, -1, nullptr, MXL_PROBS_F32, nullptr, stream, (flags & MXL_QF_SR) != 0, sr_seed,
                       (flags & MXL_QF_RHT_COL) != 0, rht_signs, qf_layout(flags));
}

extern "C" int mxl_glu_probs_quantize(const void* x_bf16, const void* probs, int probs_dtype, const uint8_t* row_mask,
                                      int64_t rows, int64_t f, int64_t row_ld, int act, int fmt, int scale_mode,
                                      const int64_t* group_lens, int num_groups, void* q_row, void* s_row, void* q_colT,
                                      void* s_colT, uint32_t flags, void* stream) {
    if (act != MXL_ACT_SILU && act != MXL_ACT_GELU) return MXL_EINVAL;
    if (probs_dtype != MXL_PROBS_F32 && probs_dtype != MXL_PROBS_BF16) return MXL_EINVAL;
    if (rows > 0 && !probs) return MXL_EINVAL;
    if (flags & ~(uint32_t)(MXL_QF_KCHUNK | MXL_QF_KSTEP | MXL_QF_KSTEP128)) return MXL_EINVAL;
    return quantize_1d(x_bf16, rows, f, row_ld, fmt, scale_mode, group_lens, num_groups, q_row, s_row, q_colT, s_colT, act,
                       probs, probs_dtype, row_mask, stream, false, 0, false, 0, qf_layout(flags));
}

extern "C" int mxl_rmsnorm_quantize(const void* x_bf16, const void* w_bf16, const void* rstd_f32, int64_t rows, int64_t k,
                                    int64_t row_ld, int fmt, int scale_mode, const int64_t* group_lens, int num_groups,
                                    void* q_row, void* s_row, void* q_colT, void* s_colT, uint32_t flags, void* stream) {
    if (!w_bf16 || (rows > 0 && !rstd_f32)) return MXL_EINVAL;
    if (flags & ~(uint32_t)(MXL_QF_KCHUNK | MXL_QF_KSTEP | MXL_QF_KSTEP128)) return MXL_EINVAL;
    return quantize_1d(x_bf16, rows, k, row_ld, fmt, scale_mode, group_lens, num_groups, q_row, s_row, q_colT, s_colT,
                       PRO_RMSNORM, rstd_f32, MXL_PROBS_F32, nullptr, stream, false, 0, false, 0,
                       qf_layout(flags), w_bf16);
}

static int quantize_weight_2d(const void* w_bf16, int64_t batch, int64_t n, int64_t k, int64_t k_ld, int64_t n_ld, int fmt,
                              int scale_mode, void* q_row, void* s_row, void* q_colT, void* s_colT, int kchunk,
                              void* stream, const void* tensor_amax = nullptr, void* scale_inv_out = nullptr,
                              const HeldQuant* pair = nullptr, bool* paired = nullptr, int parts = 1, int64_t out_rows = 0, bool keep = false) {
    if (k_ld == 0) k_ld = k;
    if (n_ld == 0) n_ld = n;
    if (out_rows == 0) out_rows = n;
    if (out_rows < n || out_rows > (n + QT - 1) / QT * QT) return MXL_EINVAL;   // the excess stays inside the last tile
    if (kchunk < 0 || (kchunk == 3 && fmt != MXL_FMT_E2M1)) return MXL_EINVAL;
    if (kchunk && ((q_row && k_ld % QT != 0) || (q_colT && n_ld % QT != 0))) return MXL_EINVAL;   // whole chunks
    if (k_ld < k || n_ld < n || k_ld % MXL_BLOCK != 0 || n_ld % MXL_BLOCK != 0) return MXL_EINVAL;
    if (n_ld > (n + QT - 1) / QT * QT) return MXL_EINVAL;  // padding of the transposed copy stays inside the last tile
    if (!w_bf16 || batch <= 0 || n <= 0 || k <= 0 || n % MXL_BLOCK != 0 || k % MXL_BLOCK != 0) return MXL_EINVAL;
    // (the transposed copy's scales may be asked for without its codes, next to a row-wise copy)
    if ((q_row == nullptr) != (s_row == nullptr) || (q_colT != nullptr && s_colT == nullptr)) return MXL_EINVAL;
    if (s_colT != nullptr && q_colT == nullptr && q_row == nullptr) return MXL_EINVAL;
    if (!q_row && !q_colT) return MXL_EINVAL;
    QuantArgs a;
    a.x = (const uint16_t*)w_bf16;
    a.rows = batch * n;
    a.cols = k;
    a.group_lens = nullptr;
    a.num_groups = 0;
    a.q_row = (uint8_t*)q_row;
    a.s_row = (uint8_t*)s_row;
    a.q_colT = (uint8_t*)q_colT;
    a.s_colT = (uint8_t*)s_colT;
    a.row_ld = k_ld;
    a.W = n_ld;  // transposed copy of each matrix is [k, n_ld]
    a.mat_rows = n;
    a.out_rows = out_rows;
    a.probs = nullptr;
    a.probs_bf16 = 0;
    a.row_mask = nullptr;
    a.norm_w = nullptr;
    a.tensor_amax = (const float*)tensor_amax;
    a.amax_parts = parts;
    a.scale_inv_out = (float*)scale_inv_out;
    a.sr_seed = 0;
    a.rht_signs = 0;
    a.kchunk = kchunk;
    a.chunk_rows_row = batch * out_rows;   // the batch is one operand of that many rows (batch * k for the transposed copy)
    a.chunk_rows_col = batch * k;
    keep_in_cache(a, keep, fmt, a.chunk_rows_row * k_ld, a.chunk_rows_col * n_ld);
    const int64_t gx = batch * ((n + QT - 1) / QT);
    const int64_t gy = ((q_row ? k_ld : k) + QT - 1) / QT;
    if (pair) {
        const QuantPairKernel kern = pair->held ? pair_kernel(*pair, fmt, tensor_amax ? SCALE_TENSOR : scale_mode, a) : nullptr;
        *paired = kern != nullptr;
        return kern ? launch_quant_pair(kern, *pair, a, gx, gy, (hipStream_t)stream) : MXL_OK;
    }
    if (tensor_amax) return dispatch_quant_tensor<true>(fmt, a, gx, gy, (hipStream_t)stream);
    return dispatch_quant<true>(fmt, scale_mode, a, gx, gy, (hipStream_t)stream);
}

namespace mxl {
int quantize_pair(const LinearOperands& o, void* stream) {
    const int lay = qf_layout(o.flags);
    const bool rht = (o.flags & MXL_QF_RHT_COL) != 0;
    auto x = [&](HeldQuant* hold) {
        return quantize_1d(o.x, o.rows, o.k, o.k_ld, o.x_fmt, o.scale_mode, o.group_lens, o.num_groups, o.xq_row, o.xs_row, o.xq_col, o.xs_col,
                           o.norm_w ? PRO_RMSNORM : -1, o.rstd, MXL_PROBS_F32, nullptr, stream, false, 0, rht, o.rht_signs, lay, o.norm_w, o.x_amax, o.x_scale_inv, hold, o.x_amax ? amax_parts(o.rows * o.k) : 1, o.keep);
    };
    auto w = [&](const HeldQuant* pair, bool* paired) {
        return quantize_weight_2d(o.w, o.batch, o.n, o.k, o.k_ld, o.n_ld, o.w_fmt, o.scale_mode, o.wq_row, o.ws_row, o.wq_col, o.ws_col, lay,
                                  stream, o.w_amax, o.w_scale_inv, pair, paired, o.w_amax ? amax_parts(o.batch * o.n * o.k) : 1, o.w_rows, o.keep);
    };
    HeldQuant hold;
    bool paired = false;
    if (o.norm_w && !o.rstd) return MXL_EINVAL;
    if (o.xq_col) {
        if (const int rc = x(&hold)) return rc;
        if (const int rc = w(&hold, &paired)) return rc;
        if (paired) return MXL_OK;
    }
    if (const int rc = x(nullptr)) return rc;
    return w(nullptr, nullptr);
}
int quantize_weight_rows(const void* w, int64_t batch, int64_t n, int64_t k, int64_t k_ld, int64_t n_ld, int64_t rows, int fmt, int scale_mode,
                         void* q_row, void* s_row, void* q_colT, void* s_colT, uint32_t flags, bool keep, void* stream) {
    return quantize_weight_2d(w, batch, n, k, k_ld, n_ld, fmt, scale_mode, q_row, s_row, q_colT, s_colT, qf_layout(flags), stream, nullptr, nullptr,
                              nullptr, nullptr, 1, rows, keep);
}
int quantize_input(const LinearInput& o, int64_t rows, int64_t cols, int64_t row_ld, int fmt, int scale_mode, const int64_t* group_lens, int num_groups,
                   void* q_row, void* s_row, void* q_colT, void* s_colT, uint32_t flags, uint64_t sr_seed, uint32_t rht_signs, bool keep, void* stream) {
    return quantize_1d(o.x, rows, cols, row_ld, fmt, scale_mode, group_lens, num_groups, q_row, s_row, q_colT, s_colT,
                       o.norm_w ? PRO_RMSNORM : o.act, o.norm_w ? o.rstd : o.probs, o.probs_dtype, o.row_mask, stream, (flags & MXL_QF_SR) != 0, sr_seed,
                       (flags & MXL_QF_RHT_COL) != 0, rht_signs, qf_layout(flags), o.norm_w, nullptr, nullptr, nullptr, 1, keep);
}
}  // namespace mxl

extern "C" int mxl_quantize_weight_2d(const void* w_bf16, int64_t batch, int64_t n, int64_t k, int64_t k_ld,
                                      int64_t n_ld, int fmt, int scale_mode, void* q_row, void* s_row, void* q_colT,
                                      void* s_colT, void* stream) {
    return quantize_weight_2d(w_bf16, batch, n, k, k_ld, n_ld, fmt, scale_mode, q_row, s_row, q_colT, s_colT, false, stream);
}

extern "C" int mxl_quantize_weight_2d_ex(const void* w_bf16, int64_t batch, int64_t n, int64_t k, int64_t k_ld,
                                         int64_t n_ld, int fmt, int scale_mode, void* q_row, void* s_row, void* q_colT,
                                         void* s_colT, uint32_t flags, void* stream) {
    if (flags & ~(uint32_t)(MXL_QF_KCHUNK | MXL_QF_KSTEP | MXL_QF_KSTEP128)) return MXL_EINVAL;
    return quantize_weight_2d(w_bf16, batch, n, k, k_ld, n_ld, fmt, scale_mode, q_row, s_row, q_colT, s_colT,
                              qf_layout(flags), stream);
}

namespace mxl {
int quantize_tensorwise_parts(const void* x, int64_t rows, int64_t cols, int64_t row_ld, int fmt, const float* amax, const int64_t* group_lens,
                              int num_groups, void* q_row, void* s_row, void* q_colT, void* s_colT, float* scale_inv, uint32_t flags,
                              void* stream) {
    return quantize_1d(x, rows, cols, row_ld, fmt, MXL_SCALE_OCP_FLOOR, group_lens, num_groups, q_row, s_row, q_colT, s_colT, -1, nullptr,
                       MXL_PROBS_F32, nullptr, stream, false, 0, false, 0, qf_layout(flags), nullptr, amax, scale_inv, nullptr,
                       amax_parts(rows * cols));
}
}  // namespace mxl

extern "C" int mxl_quantize_tensorwise(const void* x_bf16, int64_t rows, int64_t cols, int64_t row_ld, int fmt,
                                       const void* amax_f32, const int64_t* group_lens, int num_groups, void* q_row,
                                       void* s_row, void* q_colT, void* s_colT, void* scale_inv_f32, uint32_t flags,
                                       void* stream) {
    if (!amax_f32 || (fmt != MXL_FMT_E4M3 && fmt != MXL_FMT_E5M2)) return MXL_EINVAL;
    if (flags & ~(uint32_t)(MXL_QF_KCHUNK | MXL_QF_KSTEP)) return MXL_EINVAL;
    return quantize_1d(x_bf16, rows, cols, row_ld, fmt, MXL_SCALE_OCP_FLOOR, group_lens, num_groups, q_row, s_row, q_colT,
                       s_colT, -1, nullptr, MXL_PROBS_F32, nullptr, stream, false, 0, false, 0,
                       qf_layout(flags), nullptr, amax_f32, scale_inv_f32);
}

extern "C" int mxl_quantize_weight_tensorwise(const void* w_bf16, int64_t batch, int64_t n, int64_t k, int64_t k_ld,
                                              int64_t n_ld, int fmt, const void* amax_f32, void* q_row, void* s_row,
                                              void* q_colT, void* s_colT, void* scale_inv_f32, uint32_t flags,
                                              void* stream) {
    if (!amax_f32 || (fmt != MXL_FMT_E4M3 && fmt != MXL_FMT_E5M2)) return MXL_EINVAL;
    if (flags & ~(uint32_t)(MXL_QF_KCHUNK | MXL_QF_KSTEP)) return MXL_EINVAL;
    return quantize_weight_2d(w_bf16, batch, n, k, k_ld, n_ld, fmt, MXL_SCALE_OCP_FLOOR, q_row, s_row, q_colT, s_colT,
                              qf_layout(flags), stream, amax_f32, scale_inv_f32);
}

extern "C" int mxl_dequantize(const void* codes, const void* scales, int64_t rows, int64_t k, int fmt,
                              void* out_bf16, void* stream) {
    if (!codes || !scales || !out_bf16 || rows < 0 || k <= 0 || k % MXL_BLOCK != 0) return MXL_EINVAL;
    const int64_t nblocks = rows * (k / MXL_BLOCK);
    if (nblocks == 0) return MXL_OK;
    const int64_t threads = nblocks * 4;
    const int64_t grid = (threads + 255) / 256;
    if (grid > 0x7FFFFFFF) return MXL_EINVAL;
    if (fmt != MXL_FMT_E4M3 && fmt != MXL_FMT_E2M1 && fmt != MXL_FMT_E5M2) return MXL_EINVAL;
    if (!device_is_gfx950()) return MXL_ENODEV;
    if (fmt == MXL_FMT_E5M2)
        hipLaunchKernelGGL((mx_dequant_kernel<MXL_FMT_E5M2>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                           (const uint8_t*)codes, (const uint8_t*)scales, (uint16_t*)out_bf16, nblocks);
    else if (fmt == MXL_FMT_E4M3)
        hipLaunchKernelGGL((mx_dequant_kernel<MXL_FMT_E4M3>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                           (const uint8_t*)codes, (const uint8_t*)scales, (uint16_t*)out_bf16, nblocks);
    else if (fmt == MXL_FMT_E2M1)
        hipLaunchKernelGGL((mx_dequant_kernel<MXL_FMT_E2M1>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                           (const uint8_t*)codes, (const uint8_t*)scales, (uint16_t*)out_bf16, nblocks);
    else
        return MXL_EINVAL;
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}
