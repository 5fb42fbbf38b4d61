// The GEMMs of mx_gemm.hip's ring kernel on small output tiles, one workgroup per tile.
//
// The ring kernel's 256 x 256 tiles need about 256 of them before every CU has work: a linear on a few hundred tokens,
// or a weight gradient over a few hundred tokens per expert, leaves most of the chip idle (the former) or spends its
// time in prologues and epilogues that nothing overlaps (the latter: a contraction range of 256 is four K steps).
// This kernel takes the same operands (K-step-major codes and scale panels), runs the same MFMAs on every output
// element in the same order -- the results are the same bit for bit -- and differs in the split:
//   * 4 waves (2 x 2) share a TM x TN tile; two or more workgroups fit a CU, so one's epilogue and waits hide behind
//     another's MFMAs, and the hardware hands out tiles as workgroups end.  A 64 x 64 wave tile reads 2 KiB of LDS per
//     MFMA, all the LDS delivers: full chips are left to the ring kernel (4096^3: 60 us here, 56 there), while
//     [256, 4096] x [4096, 4096] takes 8.9 us instead of 41 and [64, 4096] x [14336, 4096] 13 instead of 29 (the
//     weights alone are 12 us at the rate a large copy reaches);
//   * ST LDS stages of one K step each, filled by the same LDS-direct loads; requests past the end of a contraction
//     range are sent to an offset the range check drops, so a short range moves no bytes it does not need;
//   * the group a tile belongs to is found by a wave-wide scan of group_lens.
#pragma once
#include <type_traits>

#include "mx_gemm_common.h"
#include "mx_gemm_tile.h"

namespace mxl {

constexpr int TILE_MAX_GROUPS = 256;      // four per lane in the scan

// f(0), f(1), ... f(n - 1) for a run-time n < N, each call inside the previous one's branch (no joins in between)
template <int I, int N, class F> __device__ __forceinline__ void nested_steps(int n, F&& f) {
    if constexpr (I < N - 1) {
        if (I < n) {
            f(std::integral_constant<int, I>{});
            nested_steps<I + 1, N>(n, f);
        }
    }
}

template <int TM, int TN, int ST> constexpr int tile_lds_bytes(bool b4) {
    const int loop = ST * (TM * BK + (b4 ? (TN + 127) / 128 * 4096 : TN * BK)) + 2 * (TM + TN) * 16;
    const int out = TM * (TN * 2 + 16);
    return loop > out ? loop : out;
}

template <int AFMT, int BFMT, int MODE, bool ALPHA, bool BT, int TM, int TN, int ST>
__device__ __forceinline__ void gemm_tile_body(const GemmArgs& p, uint32_t block, uint8_t* smem) {
    constexpr bool F44 = AFMT == kFmtE2M1 && BFMT == kFmtE2M1;
    constexpr bool B4 = BFMT == kFmtE2M1 && !F44;      // E2M1 weights against FP8 rows: 32 bytes per row and K step
    static_assert(AFMT != kFmtE2M1 || F44, "E2M1 rows need E2M1 columns");
    static_assert(!BT || (MODE == MODE_FWD && !B4 && TN == 128), "transposed codes: a wave's 64 columns are whole planes (or half of an E2M1 one)");
    constexpr int KS = F44 ? 2 * BK : BK;
    constexpr int PSTEPS = 512 / KS;
    constexpr int B_ROW = B4 ? BK / 2 : BK;
    constexpr int FM = TM / 64, FN = TN / 64;          // 32 x 32 fragments per wave
    constexpr int AR = TM / 64, BR = B4 ? (TN + 127) / 128 : TN / 64;   // load rounds of 4 KiB
    constexpr int R = AR + BR;
    constexpr int A_BYTES = TM * BK, STAGE = A_BYTES + BR * 4096;
    constexpr int PANEL = (TM + TN) * 16;
    constexpr int CB = BFMT == kFmtE2M1 ? 4 : BFMT == kFmtE5M2 ? 1 : 0, BL = F44 ? 4 : AFMT == kFmtE5M2 ? 1 : 0;
    constexpr uint32_t DROPPED = addr::kDropped;
    uint8_t* panels = smem + ST * STAGE;

    const int t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l = t & 63, lr = l & 31, g = l >> 5;
    const int wm = w >> 1, wn = w & 1;
    const int G = p.num_groups;
    const int tiles_n = (int)((p.n + TN - 1) / TN);

    // ---- the tile: which group, which rows, which columns ----
    uint32_t cum[TILE_MAX_GROUPS / 64], own[TILE_MAX_GROUPS / 64], tcum[TILE_MAX_GROUPS / 64], town[TILE_MAX_GROUPS / 64];
    const uint32_t cap = (uint32_t)(MODE == MODE_FWD ? p.total_m : p.k);
    int tiles_m;
    if (p.group_lens) {
        GroupScan<MODE == MODE_FWD ? 1 : MXL_SEG_ALIGN> scan(cap, G, l);
        uint32_t tbase = 0;
#pragma unroll
        for (int c = 0; c < TILE_MAX_GROUPS / 64; ++c) {
            cum[c] = tcum[c] = own[c] = town[c] = 0;
            if (c * 64 < G) {
                uint32_t end;
                scan.step(p.group_lens, c * 64, cum[c], end);
                own[c] = end - cum[c];
                // row tiles (forward) or scale panels (weight gradient) of the groups in front of this one
                town[c] = MODE == MODE_FWD ? (own[c] + TM - 1) / TM : (own[c] + 511) / 512;
                const uint32_t ts = wave_prefix(town[c]) + tbase;
                tcum[c] = ts - town[c];
                tbase = (uint32_t)__builtin_amdgcn_readlane((int)ts, 63);
            }
        }
        tiles_m = (int)tbase;
    } else {
        tiles_m = (int)((cap + TM - 1) / TM);
    }
    if (MODE == MODE_WGRAD) tiles_m = (int)((p.m + TM - 1) / TM);
    const int per_group = tiles_m * tiles_n;
    const int total = (MODE == MODE_WGRAD ? G : 1) * per_group;
    // workgroups go to the XCDs round robin: each XCD takes one contiguous run of the tile order, so that its L2 sees
    // neighbouring tiles
    const int per_xcd = (total + 7) >> 3;
    const int in_xcd = (int)(block >> 3);
    const int tile = (int)(block & 7) * per_xcd + in_xcd;
    if (in_xcd >= per_xcd || tile >= total) return;
    int grp = 0, tl = tile, pid_m, pid_n;
    if (MODE == MODE_WGRAD) {
        grp = tile / per_group;
        tl -= grp * per_group;
    }
    {
        constexpr int SUPER = 1024 / TM;                // super-rows of 1024 rows, as the ring kernel's
        const int width = SUPER * tiles_n;
        const int first = tl / width * SUPER;
        const int gsz = (tiles_m - first) < SUPER ? (tiles_m - first) : SUPER;
        pid_m = first + (tl % width) % gsz;
        pid_n = (tl % width) / gsz;
    }
    uint32_t g_row0 = 0, g_rows = cap, g_tile0 = 0;     // of the group: first row / K element, count, first row tile / panel
    if (p.group_lens) {
#pragma unroll
        for (int c = 0; c < TILE_MAX_GROUPS / 64; ++c) {
            const uint64_t hit = MODE == MODE_FWD ? __ballot(tcum[c] <= (uint32_t)pid_m && (uint32_t)pid_m < tcum[c] + town[c])
                                                  : __ballot(c * 64 + l == grp);
            if (hit) {
                const int src = __builtin_ctzll(hit);
                g_row0 = (uint32_t)__builtin_amdgcn_readlane((int)cum[c], src);
                g_rows = (uint32_t)__builtin_amdgcn_readlane((int)own[c], src);
                g_tile0 = (uint32_t)__builtin_amdgcn_readlane((int)tcum[c], src);
                if (MODE == MODE_FWD) grp = c * 64 + src;
            }
        }
    }
    int64_t a_row0, c_row0;
    int m_valid;
    uint32_t k0 = 0, kn = (uint32_t)p.k;
    if (MODE == MODE_FWD) {
        const uint32_t r = ((uint32_t)pid_m - g_tile0) * TM;
        a_row0 = (int64_t)g_row0 + r;
        m_valid = (int)(g_rows - r < TM ? g_rows - r : TM);
        c_row0 = a_row0;
    } else {
        a_row0 = (int64_t)pid_m * TM;
        m_valid = (int)((p.m - a_row0) < TM ? p.m - a_row0 : TM);
        c_row0 = (int64_t)grp * p.m + a_row0;
        k0 = g_row0;
        kn = g_rows;
    }
    const int64_t n0 = (int64_t)pid_n * TN;
    const int n_valid = (int)((p.n - n0) < TN ? p.n - n0 : TN);
    const int nst = __builtin_amdgcn_readfirstlane((int)(kn / KS));

    v16f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    if (nst > 0) {
        // ---- descriptors and per-lane offsets (addr:: as the ring kernel) ----
        const int64_t a_rows_total = MODE == MODE_FWD ? p.total_m : p.m;
        const int64_t b_rows_total = MODE == MODE_FWD ? (int64_t)G * p.b_rows : p.n;
        const int64_t bt_rows = (int64_t)G * p.k;
        const int64_t b_row0 = (MODE == MODE_FWD ? (int64_t)grp * p.b_rows : 0) + n0;
        const addr::Desc da = addr::ring_code_desc(a_rows_total, p.k / KS, a_row0, BK);
        const addr::Desc db = BT ? addr::ring_bt_desc(bt_rows, (p.n + 127) / 128 * (F44 ? 1 : 2), (int64_t)grp * p.k, (int64_t)pid_n * (F44 ? TN / 128 : TN / 64))
                                 : addr::ring_code_desc(b_rows_total, p.k / KS, b_row0, B_ROW);
        const v4i ra = make_rsrc(p.a + da.base, da.records), rb = make_rsrc(p.b + db.base, db.records);
        const uint32_t a_cstride = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a_rows_total * BK));
        const uint32_t b_cstride = BT ? (uint32_t)(KS * BK) : (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b_rows_total * B_ROW));
        const uint32_t st0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(k0 / KS));
        uint32_t va[AR], vb[BR];
#pragma unroll
        for (int e = 0; e < AR; ++e) va[e] = addr::ring_code_lane(t, e, false);
#pragma unroll
        for (int e = 0; e < BR; ++e)
            vb[e] = !BT ? addr::ring_code_lane(t, e, B4) : F44 ? addr::ring_bt4_lane(t, e, bt_rows) : addr::ring_bt_lane(t, e, bt_rows);
        // scale panels: 64 rows x 16 bytes per request, one request per wave, the row blocks of a and b dealt to the waves
        // in turn (with fewer blocks than waves some are fetched twice: every wave counts the same number of requests)
        constexpr int NB = (TM + TN) / 64;
        static_assert(NB <= 4, "one panel request per wave");
        const int64_t n_panels = (p.k + 511) / 512 + ((MODE == MODE_WGRAD && p.group_lens) ? G + 1 : 0);
        const bool is_b = w % NB >= TM / 64;
        const int blk = w % NB - (is_b ? TM / 64 : 0);
        v4i rs;
        if (!ALPHA) {
            const addr::Desc ds = is_b ? addr::ring_panel_desc(b_rows_total, n_panels, b_row0) : addr::ring_panel_desc(a_rows_total, n_panels, a_row0);
            rs = make_rsrc((is_b ? p.sb : p.sa) + ds.base, ds.records);
        }
        const uint32_t s_stride = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((is_b ? b_rows_total : a_rows_total) * 16));
        const uint32_t s_lds = (uint32_t)(uintptr_t)panels + (uint32_t)((is_b ? TM * 16 : 0) + blk * 1024);
        const uint32_t s_off = addr::ring_panel_lane(blk * 64 + l);
        const uint32_t pan0 = MODE == MODE_WGRAD ? g_tile0 * s_stride : 0u;
        const uint32_t wave_base = (uint32_t)(uintptr_t)smem + (uint32_t)(w * 1024);

        // the requests of a K step into its stage, R of them and the panel's in front; past the range they are dropped
        // but still counted
        struct Req {
            uint32_t oa, ob, base;
        };
        auto group_begin = [&](auto pan_tag, int s, int slot) __attribute__((always_inline)) {
            const bool live = s < nst;
            if constexpr (!ALPHA && decltype(pan_tag)::value)
                dma16(rs, s_lds + (uint32_t)(((s / PSTEPS) & 1) * PANEL), s_off, live ? pan0 + (uint32_t)(s / PSTEPS) * s_stride : DROPPED);
            return Req{live ? (st0 + (uint32_t)s) * a_cstride : DROPPED, live ? (BT ? (uint32_t)s : st0 + (uint32_t)s) * b_cstride : DROPPED,
                       wave_base + (uint32_t)(slot * STAGE)};
        };
        auto request = [&](auto e_tag, const Req& r) __attribute__((always_inline)) {
            constexpr int e = decltype(e_tag)::value;
            if constexpr (e < AR) dma16_at<e * 4096>(ra, r.base, va[e], r.oa);
            else dma16_at<A_BYTES + (e - AR) * 4096>(rb, r.base, vb[e - AR], r.ob);
        };

        // ---- fragment reads (64-byte rows, piece index XOR (row / 4) % 4; see the ring kernel for the BT forms) ----
        const int sw = (lr >> 2) & 3;
        const int a_frag = (wm * (TM / 2) + lr) * BK, b_frag = (wn * (TN / 2) + lr) * B_ROW;
        const int b4_lo = 16 * (g ^ ((lr >> 3) & 1));
        const int a_lo = 16 * (g ^ sw), a_hi = 16 * ((2 + g) ^ sw);
        int bt4_off[2] = {0, 0}, bt_off[2][2] = {{0, 0}, {0, 0}};
        if (BT && F44) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = 32 * g + 16 * h + (l & 15);
                bt4_off[h] = row * 64 + 16 * ((row >> 2) & 3) + 8 * ((l >> 4) & 1);
            }
        }
        if (BT && !F44) {
            const int tj = (l & 15) >> 1, ta = l & 1, tblk = (l >> 4) & 1;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    const int row = 16 * g + 8 * h + tj, cb = 32 * jj + 16 * tblk + 8 * ta;
                    bt_off[h][jj] = row * 64 + 16 * ((cb >> 4) ^ ((row >> 2) & 3)) + (cb & 15);
                }
        }
        const int a_sc = (wm * (TM / 2) + lr) * 16 + 8 * g, b_sc = TM * 16 + (wn * (TN / 2) + lr) * 16 + 8 * g;
        struct Frag {
            v8i a[FM], b[FN];
        };
        // A panel row holds [g][K step], so 8 bytes at (row, g) are a lane's scale bytes of the whole panel: two registers
        // per fragment, of which a step uses one, picking its byte with the MFMA's op_sel (no shifts).
        struct Scales {
            uint2 a[FM], b[FN];
        };
        auto read_panel = [&](Scales& sc, int pan_no) __attribute__((always_inline)) {
            const uint8_t* pan = panels + (pan_no & 1) * PANEL;
#pragma unroll
            for (int i = 0; i < FM; ++i) sc.a[i] = *(const uint2*)(pan + a_sc + i * 512);
#pragma unroll
            for (int j = 0; j < FN; ++j) sc.b[j] = *(const uint2*)(pan + b_sc + j * 512);
        };
        // fragment x of a K step: the FN fragments of b, then the FM of a
        auto read = [&](auto x_tag, Frag& f, const uint8_t* sn) __attribute__((always_inline)) {
            constexpr int x = decltype(x_tag)::value;
            if constexpr (x < FN) {
                constexpr int j = x;
                const uint8_t* r = sn + A_BYTES + b_frag + j * (32 * B_ROW);
                if constexpr (BT && F44) {
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const v2i v = __builtin_amdgcn_ds_read_tr4_b64_v2i32(
                                (__attribute__((address_space(3))) v2i*)((uint8_t*)sn + A_BYTES + q * 4096 + (bt4_off[h] ^ (16 * (wn * FN + j)))));
                            f.b[j][4 * q + 2 * h] = v[0];
                            f.b[j][4 * q + 2 * h + 1] = v[1];
                        }
                } else if constexpr (BT) {
                    static_assert(TN == 128, "a wave's 64 columns are one plane");
                    uint8_t* tb = (uint8_t*)sn + A_BYTES + wn * 4096;
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(tb + 2048 * q + bt_off[h][j]));
                            f.b[j][4 * q + 2 * h] = v[0];
                            f.b[j][4 * q + 2 * h + 1] = v[1];
                        }
                } else if constexpr (B4) {
                    const uint4 lo = *(const uint4*)(r + b4_lo);
                    f.b[j][0] = lo.x; f.b[j][1] = lo.y; f.b[j][2] = lo.z; f.b[j][3] = lo.w;
                    f.b[j][4] = 0; f.b[j][5] = 0; f.b[j][6] = 0; f.b[j][7] = 0;
                } else {
                    const uint4 lo = *(const uint4*)(r + a_lo), hi = *(const uint4*)(r + a_hi);
                    f.b[j][0] = lo.x; f.b[j][1] = lo.y; f.b[j][2] = lo.z; f.b[j][3] = lo.w;
                    f.b[j][4] = hi.x; f.b[j][5] = hi.y; f.b[j][6] = hi.z; f.b[j][7] = hi.w;
                }
            } else {
                constexpr int i = x - FN;
                const uint8_t* r = sn + a_frag + i * (32 * BK);
                const uint4 lo = *(const uint4*)(r + a_lo), hi = *(const uint4*)(r + a_hi);
                f.a[i][0] = lo.x; f.a[i][1] = lo.y; f.a[i][2] = lo.z; f.a[i][3] = lo.w;
                f.a[i][4] = hi.x; f.a[i][5] = hi.y; f.a[i][6] = hi.z; f.a[i][7] = hi.w;
            }
        };
        // MFMA x of step u of a panel
        auto multiply = [&](auto x_tag, auto u_tag, const Frag& f, const Scales& sc) __attribute__((always_inline)) {
            constexpr int j = decltype(x_tag)::value / FM, i = decltype(x_tag)::value % FM;
            constexpr int byte = (8 / PSTEPS) * decltype(u_tag)::value;
            const int sa = ALPHA ? 127 : (int)(byte < 4 ? sc.a[i].x : sc.a[i].y), sb = ALPHA ? 127 : (int)(byte < 4 ? sc.b[j].x : sc.b[j].y);
            constexpr int sel = ALPHA ? 0 : byte & 3;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.b[j], f.a[i], acc[i][j], CB, BL, sel, sb, sel, sa);
            if constexpr (F44)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                    __builtin_shufflevector(f.b[j], f.b[j], 4, 5, 6, 7, 4, 5, 6, 7), __builtin_shufflevector(f.a[i], f.a[i], 4, 5, 6, 7, 4, 5, 6, 7),
                    acc[i][j], CB, BL, sel + 1, sb, sel + 1, sa);
        };

        // ---- pipeline: ST K steps requested ahead, the fragments of step s + 1 read while step s multiplies ----
        static_for<0, ST>([&](auto s_tag) {
            constexpr int s = decltype(s_tag)::value;
            const Req r = group_begin(std::integral_constant<bool, s % PSTEPS == 0>{}, s, s);
            static_for<0, R>([&](auto e) { request(e, r); });
        });
        wait_vm<(ST - 1) * R>();
        __syncthreads();
        if (wm * (TM / 2) >= m_valid) {
            // none of this wave's rows exist (the ragged end of a group): it only keeps its share of the requests going
            int slot = 0;
            for (int s = 0; s < nst; ++s) {
                wait_vm<(ST - 2) * R>();
                __syncthreads();
                const int sn = s + ST;
                const Req r = (sn & (PSTEPS - 1)) == 0 ? group_begin(std::true_type{}, sn, slot) : group_begin(std::false_type{}, sn, slot);
                static_for<0, R>([&](auto e) { request(e, r); });
                slot = slot == ST - 1 ? 0 : slot + 1;
            }
        } else {
            Frag f0, f1;
            Scales sc;
            if (!ALPHA) read_panel(sc, 0);
            static_for<0, FM + FN>([&](auto x) { read(x, f0, smem); });
            // The waves of a workgroup come out of the barrier together: a request and a fragment read go out behind each
            // MFMA, so that the address unit and the LDS work while the MFMAs run instead of before them.  The body is
            // unrolled over whole panels and stages: stage, panel and scale byte of a step are constants, and a panel's
            // registers are loaded in straight-line code (behind a condition every step waited for its last LDS read).
            auto step = [&](auto u_tag, int s, const Frag& cur, Frag& nxt) __attribute__((always_inline)) {
                constexpr int u = decltype(u_tag)::value;
                constexpr bool LAST = (u + 1) % PSTEPS == 0;    // the panel's last step: the next one's scales are read
                wait_vm<(ST - 2) * R>();        // step s + 1 has landed
                __syncthreads();                // ... for every wave, and every wave holds the fragments of step s
                const Req r = group_begin(std::integral_constant<bool, (u + ST) % PSTEPS == 0>{}, s + ST, u % ST);
                const uint8_t* sn = smem + ((u + 1) % ST) * STAGE;
                Scales next;
                __builtin_amdgcn_sched_barrier(0);
                constexpr int NM = FM * FN, NX = FM + FN;
                static_for<0, NM>([&](auto m_tag) {
                    constexpr int m = decltype(m_tag)::value;
                    multiply(m_tag, std::integral_constant<int, u % PSTEPS>{}, cur, sc);
                    if constexpr (!ALPHA && LAST && m == 0) read_panel(next, (s + 1) / PSTEPS);
                    static_for<m * NX / NM, (m + 1) * NX / NM>([&](auto x) { read(x, nxt, sn); });   // (past the range: never multiplied)
                    static_for<m * R / NM, (m + 1) * R / NM>([&](auto e) { request(e, r); });
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (LAST) sc = next;
            };
            constexpr int UN = PSTEPS > ST ? PSTEPS : ST;
            static_assert(UN % PSTEPS == 0 && UN % ST == 0 && UN % 2 == 0, "constant stage and panel byte per unrolled step");
            auto run_step = [&](auto u_tag, int s) __attribute__((always_inline)) {
                if constexpr (decltype(u_tag)::value % 2 == 0) step(u_tag, s, f0, f1);
                else step(u_tag, s, f1, f0);
            };
            int s = 0;
            for (; s + UN <= nst; s += UN) static_for<0, UN>([&](auto u) { run_step(u, s + decltype(u)::value); });
            nested_steps<0, UN>(nst - s, [&](auto u) { run_step(u, s + decltype(u)::value); });
        }
        wait_vm<0>();
        __syncthreads();                    // nothing reads or writes the stages any more
    }

    // ---- epilogue: the tile goes through LDS (rows of TN bf16, 16 bytes of padding: conflict-free) and leaves in
    // 16-byte stores, whole rows of the tile ----
    constexpr int PITCH = TN * 2 + 16;
    float alpha = 1.f;
    if (ALPHA) alpha = *p.alpha_a * *p.alpha_b;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (ALPHA) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] *= alpha;
                }
                const v4bf o = {(__bf16)acc[i][j][4 * q], (__bf16)acc[i][j][4 * q + 1], (__bf16)acc[i][j][4 * q + 2], (__bf16)acc[i][j][4 * q + 3]};
                *(v4bf*)(smem + (wm * (TM / 2) + i * 32 + lr) * PITCH + (wn * (TN / 2) + j * 32 + 8 * q + 4 * g) * 2) = o;
            }
    __syncthreads();
    constexpr int LPR = TN / 8, RPI = 256 / LPR;       // lanes per row, rows per pass
    const int rr = t / LPR, cc = (t % LPR) * 8;
    uint16_t* ct = p.c + c_row0 * p.n + n0;
    if (cc < n_valid) {
#pragma unroll
        for (int u = 0; u < TM / RPI; ++u) {
            const int row = u * RPI + rr;
            if (row < m_valid) store16_streaming((uint8_t*)(ct + (int64_t)row * p.n + cc), *(const uint4*)(smem + row * PITCH + cc * 2));
        }
    }
}

// workgroups of a launch: the tiles there can be (a group's last row tile may be partial), a multiple of the XCDs
template <int MODE, int TM, int TN>
static int64_t tile_grid(const GemmArgs& a) {
    const int64_t tiles_n = (a.n + TN - 1) / TN;
    const int64_t tiles = MODE == MODE_WGRAD ? (int64_t)a.num_groups * ((a.m + TM - 1) / TM) * tiles_n
                          : (a.group_lens ? a.total_m / TM + a.num_groups : (a.total_m + TM - 1) / TM) * tiles_n;
    return (tiles + 7) / 8 * 8;
}

// a launch of `kern` with `lds` bytes of dynamic LDS (the attribute is set once per device and kernel)
template <class Kern, class... Args>
static int launch_tiles(Kern kern, std::atomic<bool>* attr_set, int lds, int64_t grid, hipStream_t st, const Args&... args) {
    int dev = 0;
    if (!device_is_gfx950() || hipGetDevice(&dev) != hipSuccess) return MXL_ENODEV;
    if (!attr_set[dev & 63].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return MXL_ELAUNCH;
        attr_set[dev & 63].store(true, std::memory_order_release);
    }
    if (grid <= 0) return MXL_OK;
    if (grid > 0x7FFFFFFF) return MXL_EINVAL;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, args...);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

}  // namespace mxl
