// Grouped GEMM on unquantised bf16 operands for gfx950 (v_mfma_f32_32x32x16_bf16): what the reference's grouped
// linear runs when no low-precision recipe is active -- the first / last layers of an FP4 run fall back to it --
// (primus/backends/megatron/core/extensions/primus_turbo.py:2210-2216, primus/backends/megatron/core/fp4_utils.py:155-165),
// with tokens-per-expert consumed on the device like the quantised kernels do: no host read, capturable in a graph.
//
//   forward / dgrad :  c[rows of group g, n] = a[rows of group g, k] . b_g^T        b_g = [n, k]   (contraction contiguous)
//                                                                   or . b_g          b_g = [k, n]   (MXL_BF_B_KN)
//   wgrad           :  c[g][m_out, n_out] = sum over the tokens t of group g of p[t, m_out] * q[t, n_out]
//
// Two kernels, chosen per launch, 256 output columns per tile each: 256 rows (bf16_gemm_tall_kernel: 8 waves, one
// workgroup per CU) and, for forward / dgrad over groups of fewer rows, where a 256-row tile would mostly hold padding,
// 128 rows (bf16_gemm_kernel: 4 waves of 64 x 128, two workgroups per CU, two stages of 32 contraction elements).  Both
// fill LDS by LDS-direct loads (buffer_load ... lds).  An operand whose contraction dim is contiguous in memory is
// staged by rows and read with ds_read_b128; one whose contraction dim is the slow one (the [k, n] weight, both
// operands of wgrad) is staged as it lies, [contraction][columns], and read with the transposing LDS read ds_read_b64_tr_b16,
// which hands every lane four consecutive contraction elements of its own column.  Measured lane mapping of that
// read: inside each block of 16 lanes, lane 4 a + e receives element e of the 8-byte pieces addressed by lanes a,
// a + 4, a + 8, a + 12 (in this order).  16-byte pieces are XOR-swizzled on the global side so that both kinds of
// read are spread over the LDS banks.  The tile list is derived from group_lens by every workgroup; the workgroups
// are persistent and walk it in rounds.  Both kernels add every output element's products in the same order: the same bits.
#include "mx_device.h"
#include "mx_gemm_addr.h"

#include <type_traits>

namespace mxl {

constexpr int BF_BN = 256;
constexpr int BF_KS = 32;                  // contraction elements per slot (two MFMA K steps of 16)
constexpr int BF_THREADS = 256;
constexpr int BF_B_BYTES = BF_BN * 64;     // 16 KiB of b per stage; a: BM * 64
constexpr int BF_CPITCH = 264;             // bytes per staged output row: 128 bf16 + 8 (rows spread over the banks)
constexpr int BF_GROUP_M = 8;              // tile order: super-rows of this many row tiles

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Bf16Args {
    const uint8_t* a;      // forward: activations [total_m, k];   wgrad: p [total_m, m_out]
    const uint8_t* b;      // forward: weights [G, n, k] or [G, k, n];   wgrad: q [total_m, n_out]
    void* c;
    const int64_t* group_lens;
    int num_groups;
    int64_t total_m;
    int64_t m;             // wgrad: m_out
    int64_t n;             // forward: n;  wgrad: n_out
    int64_t k;             // forward: contraction length
};

__device__ __forceinline__ v4i bf_rsrc(const void* base, int64_t bytes) {
    const uint64_t p = (uint64_t)base;
    const uint32_t n = bytes > 0xFFFFFFFFll ? 0xFFFFFFFFu : (uint32_t)(bytes < 0 ? 0 : bytes);
    v4i r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32) & 0xFFFF);
    r[2] = __builtin_amdgcn_readfirstlane((int)n);     // the range check covers per-lane + scalar offset: past it, zeros
    r[3] = 0x00020000;
    return r;
}
__device__ __forceinline__ v4i bf_desc(const uint8_t* operand, const addr::Desc& d) { return bf_rsrc(operand + d.base, d.records); }
// LDS-direct 16-byte load: lane i's data lands at lds_off + 16 i.  (M0 holds nothing else in this kernel.)
__device__ __forceinline__ void bf_dma16(v4i rsrc, uint32_t lds_off, uint32_t voff, uint32_t soff) {
    asm volatile("" : "+s"(soff));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_off), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

// the same with the LDS address formed in the request's own scalar instruction (base + constant): two scalar
// instructions per request instead of five
template <int LDS_IMM>
__device__ __forceinline__ void bf_dma16_at(v4i rsrc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                 :
                 : "s"(lds_base), "n"(LDS_IMM), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "scc");
}

// one dword per lane into LDS: the line it lies in is in the L2 afterwards
__device__ __forceinline__ void bf_dma4(v4i rsrc, uint32_t lds_off, uint32_t voff, uint32_t soff) {
    asm volatile("" : "+s"(soff));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(lds_off), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

constexpr int bf16_lds_bytes() {
    return 2 * (128 * 64 + BF_B_BYTES) + (MXL_MAX_GROUPS + 2) * 4 + (MXL_MAX_GROUPS + 2) * 8;
}
template <int N>
__device__ __forceinline__ void bf_wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// prefix sums over the groups of their rows and of their row tiles; lens clamped to what the buffers hold
template <int BM>
__device__ __forceinline__ void bf16_group_table(const Bf16Args& p, int64_t* pre_rows, int* pre_tiles, int t) {
    if (t < 64) {
        GroupScan<> scan(p.total_m, p.num_groups, t);
        uint32_t tiles = 0;
        if (t == 0) pre_tiles[0] = 0, pre_rows[0] = 0;
        for (int c = 0; c < p.num_groups; c += 64) {
            uint32_t first, end;
            scan.step(p.group_lens, c, first, end);
            const uint32_t te = wave_prefix((end - first + BM - 1) / BM) + tiles;
            if (c + t < p.num_groups) pre_tiles[c + t + 1] = (int)te, pre_rows[c + t + 1] = end;
            tiles = (uint32_t)__builtin_amdgcn_readlane((int)te, 63);
        }
    }
    __syncthreads();
}
// a fragment's 8 contraction elements of step ks from an operand staged [contraction row][256 columns]
__device__ __forceinline__ v8bf bf16_read_trans(uint8_t* lane, int ks) {
    v8bf out;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)(lane + ks * 8192 + h * 2048));
        const v4bf q = __builtin_bit_cast(v4bf, v);
        out[4 * h] = q[0]; out[4 * h + 1] = q[1]; out[4 * h + 2] = q[2]; out[4 * h + 3] = q[3];
    }
    return out;
}

// A_T / B_T: the operand's contraction dim is the slow one in memory (staged [32][cols], transposing reads).
// WGRAD: contraction over the tokens of a group (both operands A_T / B_T), one output matrix per group.
// ACCUM (wgrad): c is float32 and the result is added to it.
template <bool A_T, bool B_T, bool WGRAD, bool ACCUM>
__global__ __launch_bounds__(BF_THREADS, 2) void bf16_gemm_kernel(Bf16Args p) {
    static_assert(!WGRAD || (A_T && B_T), "wgrad contracts over tokens: both operands are token-major");
    static_assert(!ACCUM || WGRAD, "only the weight gradient accumulates");
    constexpr int BF_BM = 128, NST = 2;
    constexpr int BF_A_BYTES = BF_BM * 64, BF_STAGE = BF_A_BYTES + BF_B_BYTES;
    constexpr int MI = BF_BM / 64;             // 32-row fragments per wave
    constexpr int AR = BF_BM / 64;             // load rounds of 4 KiB for a (b: 4)
    constexpr int LOADS = AR + 4;              // requests per wave and slot
    static_assert(BF_BM * BF_CPITCH <= NST * BF_STAGE, "the output staging area reuses the operand stages");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int* pre_tiles = (int*)(smem + NST * BF_STAGE);
    int64_t* pre_rows = (int64_t*)(pre_tiles + MXL_MAX_GROUPS + 2);
    const int t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l = t & 63, lr = l & 31, g = l >> 5;
    const int wm = w >> 1, wn = w & 1;
    const int G = p.num_groups;
    const uint32_t smem_base = (uint32_t)(uintptr_t)smem;

    bf16_group_table<BF_BM>(p, pre_rows, pre_tiles, t);

    const int tiles_n = (int)((p.n + BF_BN - 1) / BF_BN);
    const int tiles_m = WGRAD ? (int)((p.m + BF_BM - 1) / BF_BM) : pre_tiles[G];
    const int total_tiles = WGRAD ? G * tiles_m * tiles_n : tiles_m * tiles_n;
    // Persistent workgroups (one per CU for the 256-row tile, two for the 128-row one) walk the tile order in rounds:
    // every workgroup starts its tile of a round at the same time and all tiles of a launch have the same contraction
    // length, so the 32 tiles an XCD works on stay within a few K slots of each other and share their operand panels
    // through that XCD's L2 (with one workgroup per tile, started whenever a CU fell free, the tiles of an XCD drifted
    // apart and the launch filled the L2s with 1.75 times the bytes).  Consecutive workgroup ids land on different XCDs:
    // XCD x takes the x-th run of gridDim / 8 tiles of every round.
    const int nwg = gridDim.x;
    const int vwg = (nwg & 7) ? (int)blockIdx.x : ((int)(blockIdx.x & 7) * (nwg >> 3) + (int)(blockIdx.x >> 3));
  for (int tile_id = vwg; tile_id < total_tiles; tile_id += nwg) {
    int tile = tile_id;
    int grp = 0;
    if (WGRAD) {
        grp = tile / (tiles_m * tiles_n);
        tile -= grp * tiles_m * tiles_n;
    }
    int pid_m, pid_n;
    {
        const int width = BF_GROUP_M * tiles_n;
        const int first = (tile / width) * BF_GROUP_M;
        const int gsz = (tiles_m - first) < BF_GROUP_M ? (tiles_m - first) : BF_GROUP_M;
        pid_m = first + (tile % width) % gsz;
        pid_n = (tile % width) / gsz;
    }
    const int64_t n0 = (int64_t)pid_n * BF_BN;
    const int n_valid = (p.n - n0) < BF_BN ? (int)(p.n - n0) : BF_BN;
    int m_valid, nslots;
    int64_t c_row0;                 // first output row (forward: token row; wgrad: row inside the group's matrix)
    v4i ra, rb;
    uint32_t a_step, b_step;        // bytes from one K slot to the next
    uint32_t va[AR], vb[4];         // per-lane offsets of the load rounds
    if (!WGRAD) {
        int lo = 0, hi = G;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (pre_tiles[mid] <= pid_m) lo = mid; else hi = mid;
        }
        grp = lo;
        const int64_t g_row0 = pre_rows[grp], g_rows = pre_rows[grp + 1] - g_row0;
        const int64_t r = (int64_t)(pid_m - pre_tiles[grp]) * BF_BM;
        c_row0 = g_row0 + r;
        m_valid = (g_rows - r) < BF_BM ? (int)(g_rows - r) : BF_BM;
        nslots = (int)(p.k / BF_KS);
        // a: [total_m, k], contraction contiguous; rows past the operand's end are dropped by the range check
        const int64_t lda = p.k * 2;
        ra = bf_rsrc(p.a + c_row0 * lda, (p.total_m - c_row0) * lda);
        a_step = 64;
#pragma unroll
        for (int e = 0; e < AR; ++e) {
            const int row = (t >> 2) + 64 * e;
            va[e] = (uint32_t)(row * lda + 16 * ((t & 3) ^ ((row >> 2) & 3)));
        }
        if (!B_T) {
            const int64_t ldb = p.k * 2, b_row0 = (int64_t)grp * p.n + n0;
            rb = bf_rsrc(p.b + b_row0 * ldb, ((int64_t)G * p.n - b_row0) * ldb);
            b_step = 64;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (t >> 2) + 64 * e;
                vb[e] = (uint32_t)(row * ldb + 16 * ((t & 3) ^ ((row >> 2) & 3)));
            }
        } else {
            // b_g: [k, n]: 32 contraction rows of 512 bytes per slot; the descriptor ends with the group's matrix
            const int64_t ldb = p.n * 2;
            rb = bf_rsrc(p.b + ((int64_t)grp * p.k * p.n + n0) * 2, (p.k * p.n - n0) * 2);
            b_step = (uint32_t)(BF_KS * ldb);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (t >> 5) + 8 * e;
                vb[e] = (uint32_t)(row * ldb + 16 * ((t & 31) ^ ((row & 3) << 2)));
            }
        }
    } else {
        const int64_t m0 = (int64_t)pid_m * BF_BM;
        c_row0 = m0;
        m_valid = (p.m - m0) < BF_BM ? (int)(p.m - m0) : BF_BM;
        const int64_t t0 = pre_rows[grp], len = pre_rows[grp + 1] - t0;
        nslots = (int)((len + BF_KS - 1) / BF_KS);
        // p: [total_m, m_out], q: [total_m, n_out], token-major; the descriptors end with the group's last token, so
        // the rows of a partly filled last slot read as zero
        const int64_t lda = p.m * 2, ldb = p.n * 2;
        ra = bf_rsrc(p.a + t0 * lda + m0 * 2, len * lda - m0 * 2);
        rb = bf_rsrc(p.b + t0 * ldb + n0 * 2, len * ldb - n0 * 2);
        a_step = (uint32_t)(BF_KS * lda);
        b_step = (uint32_t)(BF_KS * ldb);
        // a round of 4 KiB holds 32 / AR contraction rows of BM columns
#pragma unroll
        for (int e = 0; e < AR; ++e) {
            const int row = t / (BF_BM / 8) + (32 / AR) * e;
            va[e] = (uint32_t)(row * lda + 16 * ((t % (BF_BM / 8)) ^ ((row & 3) << 2)));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = (t >> 5) + 8 * e;
            vb[e] = (uint32_t)(row * ldb + 16 * ((t & 31) ^ ((row & 3) << 2)));
        }
    }
    a_step = (uint32_t)__builtin_amdgcn_readfirstlane((int)a_step);
    b_step = (uint32_t)__builtin_amdgcn_readfirstlane((int)b_step);
    nslots = __builtin_amdgcn_readfirstlane(nslots);

    auto issue = [&](int slot, int stage) __attribute__((always_inline)) {
        const uint32_t base = smem_base + (uint32_t)(stage * BF_STAGE) + (uint32_t)(w * 1024);
        const uint32_t sa = (uint32_t)slot * a_step, sb = (uint32_t)slot * b_step;
#pragma unroll
        for (int e = 0; e < AR; ++e) bf_dma16(ra, base + e * 4096, va[e], sa);
#pragma unroll
        for (int e = 0; e < 4; ++e) bf_dma16(rb, base + BF_A_BYTES + e * 4096, vb[e], sb);
    };

    // ---- per-lane constants of the fragment reads ----
    // contiguous operand, 64-byte rows: lane (row lr, half g) reads piece 2 ks + g, XOR (row / 4) % 4
    const int ca_row = wm * (BF_BM / 2) + lr, cb_row = wn * 128 + lr;
    // transposed operand: this lane ADDRESSES row j of a 4-row group, 8-byte piece `a4` of its 16-lane block's 16 columns
    const int tj = (l & 15) >> 2, ta4 = l & 3, tblk = (l >> 4) & 1;
    const int t_colbyte = 32 * tblk + 8 * ta4;     // byte offset of the piece inside a 32-column fragment

    v16f acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    auto read_contig = [&](const uint8_t* base, int row, int ks) __attribute__((always_inline)) {
        return *(const v8bf*)(base + row * 64 + 16 * ((2 * ks + g) ^ ((row >> 2) & 3)));
    };
    // pitch: bytes per staged contraction row (256 for the 128-wide operand, 512 for the 256-wide one); col0: first
    // column of the fragment inside the tile
    auto read_trans = [&](uint8_t* base, int pitch, int col0, int ks) __attribute__((always_inline)) {
        v8bf out;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 16 * ks + 8 * g + 4 * h + tj;
            const int byte = 2 * col0 + t_colbyte;
            uint8_t* ptr = base + row * pitch + 16 * ((byte >> 4) ^ ((row & 3) << 2)) + (byte & 15);
            const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)ptr);
            const v4bf vb4 = __builtin_bit_cast(v4bf, v);
            out[4 * h] = vb4[0]; out[4 * h + 1] = vb4[1]; out[4 * h + 2] = vb4[2]; out[4 * h + 3] = vb4[3];
        }
        return out;
    };

    // does this wave hold rows of the tile?  (if not it only keeps the requests going)
    const bool live = __builtin_amdgcn_readfirstlane(m_valid > wm * (BF_BM / 2));

    auto read_a = [&](uint8_t* sa, int i, int ks) __attribute__((always_inline)) {
        return A_T ? read_trans(sa, BF_BM * 2, wm * (BF_BM / 2) + 32 * i, ks) : read_contig(sa, ca_row + 32 * i, ks);
    };
    auto read_b = [&](uint8_t* sb, int j, int ks) __attribute__((always_inline)) {
        return B_T ? read_trans(sb, 512, wn * 128 + 32 * j, ks) : read_contig(sb, cb_row + 32 * j, ks);
    };
    if (nslots > 0) issue(0, 0);
    for (int s = 0; s < nslots; ++s) {
        bf_wait_vm<0>();
        __syncthreads();     // slot s is in LDS for every wave, and every wave has left the stage of slot s - 1
        if (s + 1 < nslots) issue(s + 1, (s + 1) & 1);
        uint8_t* sa = smem + (s & 1) * BF_STAGE;
        uint8_t* sb = sa + BF_A_BYTES;
        if (!live) continue;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            v8bf fb[4], fa[MI];
#pragma unroll
            for (int j = 0; j < 4; ++j) fb[j] = read_b(sb, j, ks);
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[i] = read_a(sa, i, ks);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();         // every wave is done with the stages: they become the output staging area

    // lane (lr, g) of fragment (i, j) holds row 32 i + lr, columns 32 j + 8 q + 4 g .. + 3 in registers 4 q .. 4 q + 3
    if (ACCUM) {
        float* c = (float*)p.c + ((int64_t)grp * p.m + c_row0) * p.n + n0;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int row = wm * (BF_BM / 2) + 32 * i + lr;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int col = wn * 128 + 32 * j + 8 * q + 4 * g;
                    if (row < m_valid && col < n_valid) {      // n_out is a multiple of 8: a quad is in or out as a whole
                        v4f* dst = (v4f*)(c + (int64_t)row * p.n + col);
                        v4f o = *dst;
                        o[0] += acc[i][j][4 * q]; o[1] += acc[i][j][4 * q + 1]; o[2] += acc[i][j][4 * q + 2]; o[3] += acc[i][j][4 * q + 3];
                        *dst = o;
                    }
                }
        }
    } else {
        uint16_t* c = (uint16_t*)p.c + ((WGRAD ? (int64_t)grp * p.m : 0) + c_row0) * p.n + n0;
        // two passes, one per 128-column half: its waves stage BM x 128 bf16, then all threads store whole rows
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h) __syncthreads();
            if (wn == h) {
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const v4bf o = {(__bf16)acc[i][j][4 * q], (__bf16)acc[i][j][4 * q + 1], (__bf16)acc[i][j][4 * q + 2],
                                            (__bf16)acc[i][j][4 * q + 3]};
                            *(v4bf*)(smem + (wm * (BF_BM / 2) + 32 * i + lr) * BF_CPITCH + (32 * j + 8 * q + 4 * g) * 2) = o;
                        }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < BF_BM / 16; ++u) {
                const int idx = u * BF_THREADS + t, row = idx >> 4, piece = idx & 15;
                const int col = h * 128 + piece * 8;
                if (row < m_valid && col < n_valid) {
                    const uint2 lo = *(const uint2*)(smem + row * BF_CPITCH + piece * 16);      // rows are 8-byte aligned
                    const uint2 hi = *(const uint2*)(smem + row * BF_CPITCH + piece * 16 + 8);
                    *(uint4*)(c + (int64_t)row * p.n + col) = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
            }
        }
    }
    __syncthreads();         // every wave has left the staging area: the next tile's requests may overwrite it
  }
}

// ---- the 256-row tile: 8 waves (2 x 4) of 128 x 64, two per SIMD, K slots of 64 elements ----
// Bound by the board's power limit where the groups are long (MFMA busy 0.80 at 1.55 GHz; the vendor library's dense
// kernel on the same problem 0.88 at 1.51, 7 % faster), by the padding of the groups' last tiles where they are short.
// What the split is for:
//   * two waves per SIMD: one's requests, reads and barriers run under the other's MFMAs.  Four waves of 128 x 128, one
//     per SIMD, had MFMA busy 0.58 whatever the order of their instructions;
//   * slots of 64 elements: a request moves whole 128-byte lines of a contiguous operand (32 elements: half lines);
//   * requests close behind the barrier that frees their stage (spread over 15 MFMAs; over 22: -3 %, over 30: -6 %): they
//     have one slot, about a microsecond, to land;
//   * the L2 is asked four slots ahead for the lines this tile's neighbours on the XCD will want, each line by one of
//     them: a fifth of the requests missed the L2 and every slot waited for some of those (-15 % cycles);
//   * the next tile's first slot is requested in front of the output's way out (wgrad of 1000 tokens: +1.5 %).
// Against its 4-wave predecessor (wgrad: the 128-row tile it ran on), ragged groups, forward / dgrad / wgrad in PFLOP/s:
// Mixtral experts [32768, 4096] x [8, 28672, 4096] 1.04 / 1.03 / 1.12 -> 1.23 / 1.12 / 1.28; 32 groups of about 1024 rows,
// [4096, 7168], 0.89 / 0.94 / 0.96 -> 1.07 / 1.09 / 1.09; 128 groups of about 512, [5760, 2880], 0.68 / 0.78 / 0.75 ->
// 0.87 / 0.86 / 0.81.  (At the power limit the rate follows the box and the data: up to 1.27 / 1.30 / 1.36 on the first.)
constexpr int TL_THREADS = 512;
constexpr int TL_KS = 64;                               // contraction elements per slot: 128 bytes of a row, four MFMA steps
constexpr int TL_HALF = 256 * TL_KS * 2;                // 32 KiB: one operand of a slot
constexpr int TL_STAGE = 2 * TL_HALF, TL_OPS = 2;       // two stages
constexpr int TL_REQ = 8;                               // requests per wave and slot: four rounds of 8 KiB per operand
constexpr int TL_AHEAD = 4;                             // slots the L2 is asked ahead
constexpr int TL_TABLES = (MXL_MAX_GROUPS + 2) * 4 + (MXL_MAX_GROUPS + 2) * 8;
constexpr int tall_lds_bytes() { return TL_OPS * TL_STAGE + TL_TABLES + 256; }      // (256: where the L2 requests' dwords land)

template <int I, int N, class F>
__device__ __forceinline__ void bf_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        bf_static_for<I + 1, N>(f);
    }
}

template <bool A_T, bool B_T, bool WGRAD, bool ACCUM>
__global__ __launch_bounds__(TL_THREADS, 2) void bf16_gemm_tall_kernel(Bf16Args p) {
    static_assert(!WGRAD || (A_T && B_T), "wgrad contracts over tokens: both operands are token-major");
    static_assert(!ACCUM || WGRAD, "only the weight gradient accumulates");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int* pre_tiles = (int*)(smem + TL_OPS * TL_STAGE);
    int64_t* pre_rows = (int64_t*)(pre_tiles + MXL_MAX_GROUPS + 2);
    const int t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l = t & 63, lr = l & 31, g = l >> 5;
    const int wm = w >> 2, wn = w & 3;      // the two waves of a SIMD hold different rows: a tile of <= 128 rows keeps one busy on each
    const int G = p.num_groups;
    const uint32_t smem_base = (uint32_t)(uintptr_t)smem;
    bf16_group_table<256>(p, pre_rows, pre_tiles, t);

    const int tiles_n = (int)((p.n + BF_BN - 1) / BF_BN);
    const int tiles_m = WGRAD ? (int)((p.m + 255) / 256) : pre_tiles[G];
    const int total_tiles = WGRAD ? G * tiles_m * tiles_n : tiles_m * tiles_n;
    const int nwg = gridDim.x;
    const int vwg = (nwg & 7) ? (int)blockIdx.x : ((int)(blockIdx.x & 7) * (nwg >> 3) + (int)(blockIdx.x >> 3));

    // ---- per-lane constants ----
    // fragment reads: contiguous, row lr of a fragment, piece 2 ks + g XOR (row / 2) % 8 (16 lanes are served at a time,
    // 256 bytes: 16 rows have to put the piece into 16 different places of two rows; with row % 8 half of them met)
    const int lane_c = lr * 128 + 16 * (g ^ ((lr >> 1) & 7));
    const int a_c = wm * 128 * 128 + lane_c, b_c = TL_HALF + wn * 64 * 128 + lane_c;
    // transposed: this lane addresses row tj of a 4-row group, 8-byte piece ta4 of its 16-lane block's 16 columns
    const int tj = (l & 15) >> 2, ta4 = l & 3, tblk = (l >> 4) & 1;
    const int lane_t = (8 * g + tj) * 512 + 8 * (ta4 & 1), t_col16 = 2 * tblk + (ta4 >> 1);

    struct Tile {
        int64_t n0, c_row0;             // first output column and row (forward: token row; wgrad: row inside the group's matrix)
        int grp, m_valid, n_valid;
        int halves;                     // contraction in halves of a slot (32 elements)
        uint32_t a_step, b_step;        // bytes from one K slot to the next
        v4i ra, rb;
        uint32_t va[4], vb[4];          // per-lane offsets of the load rounds
        v4i rp;                         // the L2 request: descriptor, bytes from slot to slot, per-lane offset
        uint32_t p_step, vp;
    };
    auto setup = [&](int tile) __attribute__((always_inline)) {
        Tile q;
        int grp = 0;
        if (WGRAD) {
            grp = tile / (tiles_m * tiles_n);
            tile -= grp * tiles_m * tiles_n;
        }
        int pid_m, pid_n;
        {
            const int width = BF_GROUP_M * tiles_n;
            const int first = (tile / width) * BF_GROUP_M;
            const int gsz = (tiles_m - first) < BF_GROUP_M ? (tiles_m - first) : BF_GROUP_M;
            pid_m = first + (tile % width) % gsz;
            pid_n = (tile % width) / gsz;
        }
        const int64_t n0 = (int64_t)pid_n * BF_BN;
        const int n_valid = (p.n - n0) < BF_BN ? (int)(p.n - n0) : BF_BN;
        int64_t klen, c_row0;
        int m_valid;
        uint32_t a_step, b_step;
        if (!WGRAD) {
            int lo = 0, hi = G;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (pre_tiles[mid] <= pid_m) lo = mid; else hi = mid;
            }
            grp = lo;
            const int64_t g_row0 = pre_rows[grp], g_rows = pre_rows[grp + 1] - g_row0;
            const int64_t r = (int64_t)(pid_m - pre_tiles[grp]) * 256;
            c_row0 = g_row0 + r;
            m_valid = (g_rows - r) < 256 ? (int)(g_rows - r) : 256;
            klen = p.k;
            const int64_t lda = p.k * 2;
            q.ra = bf_desc(p.a, addr::tall_rows_desc(p.total_m, c_row0, lda));
            a_step = TL_KS * 2;
#pragma unroll
            for (int e = 0; e < 4; ++e) q.va[e] = addr::tall_rows_lane(t, e, lda);
            if (!B_T) {
                const int64_t ldb = p.k * 2, b_row0 = (int64_t)grp * p.n + n0;
                q.rb = bf_desc(p.b, addr::tall_rows_desc((int64_t)G * p.n, b_row0, ldb));
                b_step = TL_KS * 2;
#pragma unroll
                for (int e = 0; e < 4; ++e) q.vb[e] = addr::tall_rows_lane(t, e, ldb);
            } else {
                const int64_t ldb = p.n * 2;
                q.rb = bf_desc(p.b, addr::tall_cols_desc(grp * p.k, p.k, ldb, n0 * 2));
                b_step = (uint32_t)(TL_KS * ldb);
#pragma unroll
                for (int e = 0; e < 4; ++e) q.vb[e] = addr::tall_cols_lane(t, e, ldb);
            }
        } else {
            const int64_t m0 = (int64_t)pid_m * 256;
            c_row0 = m0;
            m_valid = (p.m - m0) < 256 ? (int)(p.m - m0) : 256;
            const int64_t t0 = pre_rows[grp];
            klen = pre_rows[grp + 1] - t0;
            // the descriptors end with the group's last token: the rows of a partly filled last slot read as zero
            const int64_t lda = p.m * 2, ldb = p.n * 2;
            q.ra = bf_desc(p.a, addr::tall_cols_desc(t0, klen, lda, m0 * 2));
            q.rb = bf_desc(p.b, addr::tall_cols_desc(t0, klen, ldb, n0 * 2));
            a_step = (uint32_t)(TL_KS * lda);
            b_step = (uint32_t)(TL_KS * ldb);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                q.va[e] = addr::tall_cols_lane(t, e, lda);
                q.vb[e] = addr::tall_cols_lane(t, e, ldb);
            }
        }
        q.a_step = (uint32_t)__builtin_amdgcn_readfirstlane((int)a_step);
        q.b_step = (uint32_t)__builtin_amdgcn_readfirstlane((int)b_step);
        {
            // lines of 128 bytes this tile asks the L2 for: a quarter of a's 256 of a slot (waves 0 .. 3, 16 lanes each),
            // an eighth of b's (waves 4 .. 7, 8 lanes).  Rows of a at a power of two apart are left out (an empty
            // descriptor drops the request): asking for them costs more than it gives (k = 4096: 1.17 with, 1.22 without).
            const bool of_a = w < 4, trans = of_a ? A_T : B_T;
            const int line = of_a ? (pid_n & 3) * 64 + w * 16 + (l & 15) : (pid_m & 7) * 32 + (w - 4) * 8 + (l & 7);
            const int64_t ld = (of_a ? (WGRAD ? p.m : p.k) : (WGRAD || B_T ? p.n : p.k)) * 2;
            const bool ask = trans || !of_a || (ld & (ld - 1)) != 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) q.rp[i] = __builtin_amdgcn_readfirstlane(of_a ? q.ra[i] : q.rb[i]);
            if (!ask) q.rp[2] = 0;
            q.p_step = (uint32_t)__builtin_amdgcn_readfirstlane(ask ? (int)(of_a ? a_step : b_step) : 0);
            q.vp = addr::tall_l2_lane(line, trans, ld);
        }
        q.halves = __builtin_amdgcn_readfirstlane((int)((klen + 31) / 32));
        q.m_valid = __builtin_amdgcn_readfirstlane(m_valid);
        q.n_valid = n_valid;
        q.grp = grp;
        q.n0 = n0;
        q.c_row0 = c_row0;
        return q;
    };
    // requests of a slot; past the last slot the descriptors are empty, so the range check drops them
    struct In {
        v4i ra, rb;
        uint32_t base, sa, sb;
    };
    auto in_begin = [&](const Tile& q, int slot) __attribute__((always_inline)) {
        In r{q.ra, q.rb, smem_base + (uint32_t)((slot & 1) * TL_STAGE) + (uint32_t)(w * 1024), (uint32_t)slot * q.a_step, (uint32_t)slot * q.b_step};
        if (2 * slot >= q.halves) r.ra[2] = 0, r.rb[2] = 0, r.sa = 0, r.sb = 0;
        return r;
    };
    auto request = [&](auto e_tag, const In& r, const Tile& q) __attribute__((always_inline)) {
        constexpr int e = decltype(e_tag)::value;       // the operands in turn
        if constexpr ((e & 1) == 0) bf_dma16_at<(e >> 1) * 8192>(r.ra, r.base, q.va[e >> 1], r.sa);
        else bf_dma16_at<TL_HALF + (e >> 1) * 8192>(r.rb, r.base, q.vb[e >> 1], r.sb);
    };
    const uint32_t ahead_lds = smem_base + TL_OPS * TL_STAGE + TL_TABLES;
    auto ask_l2 = [&](const Tile& q, int slot) __attribute__((always_inline)) {
        v4i r = q.rp;
        uint32_t so = (uint32_t)slot * q.p_step;
        if (2 * slot >= q.halves) r[2] = 0, so = 0;
        if (l < (w < 4 ? 16 : 8)) bf_dma4(r, ahead_lds, q.vp, so);
    };
    auto first_slot = [&](const Tile& q) __attribute__((always_inline)) {
        const In r = in_begin(q, 0);
        bf_static_for<0, TL_REQ>([&](auto e) { request(e, r, q); });
    };

    if (vwg >= total_tiles) return;
    Tile tl = setup(vwg);
    first_slot(tl);
    for (int tile_id = vwg;;) {
        // an odd half is the first half of a last slot (what lies past it in the slot belongs to the next row and is not
        // multiplied)
        const int halves = tl.halves, nfull = halves >> 1;
        v16f acc[4][2];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

        // row fragments of this wave that hold rows of the tile
        int live = (tl.m_valid - wm * 128 + 31) >> 5;
        live = live < 0 || wn * 64 >= tl.n_valid ? 0 : live;

        auto read_a = [&](uint8_t* st, auto i_tag, auto ks_tag) __attribute__((always_inline)) {
            constexpr int i = decltype(i_tag)::value, ks = decltype(ks_tag)::value;
            if constexpr (!A_T) return *(const v8bf*)(st + (a_c ^ (32 * ks)) + i * 4096);
            else return bf16_read_trans(st + lane_t + 16 * ((16 * wm + 4 * i + t_col16) ^ (tj << 2)), ks);
        };
        auto read_b = [&](uint8_t* st, auto j_tag, auto ks_tag) __attribute__((always_inline)) {
            constexpr int j = decltype(j_tag)::value, ks = decltype(ks_tag)::value;
            if constexpr (!B_T) return *(const v8bf*)(st + (b_c ^ (32 * ks)) + j * 4096);
            else return bf16_read_trans(st + TL_HALF + lane_t + 16 * ((8 * wn + 4 * j + t_col16) ^ (tj << 2)), ks);
        };

        // One MFMA step (16 elements) multiplies while the next one's fragments are read; every read and request sits
        // between two MFMAs (pinned).  The slot's barrier stands one MFMA into its last step: by then every wave holds
        // all its fragments of the slot, so the stage is free for the slot after next, whose requests are spread over
        // the rest of this step and the next one.  With two waves per SIMD one's barrier and waits run under the other's MFMAs.
        auto run = [&](auto live_tag) __attribute__((always_inline)) {
            constexpr int L = decltype(live_tag)::value;
            constexpr int NM = 2 * L, NR = L + 2, NB = 1;             // MFMAs, reads per step; MFMAs in front of the barrier
            constexpr int Q = (NM - NB) + NM;                         // gaps the requests are spread over
            constexpr int E3 = (NM - NB) * TL_REQ / Q;                // of them behind the barrier of the slot
            In in = in_begin(tl, 1);
            bf_static_for<0, E3>([&](auto e) { request(e, in, tl); });
            bf_wait_vm<E3>();
            __syncthreads();
            v8bf fa[2][L], fb[2][2];
            auto read = [&](auto x_tag, auto ks_tag, uint8_t* st) __attribute__((always_inline)) {
                constexpr int x = decltype(x_tag)::value, ks = decltype(ks_tag)::value;
                if constexpr (x == 0) fb[ks & 1][0] = read_b(st, std::integral_constant<int, 0>{}, ks_tag);
                else if constexpr (x <= L) fa[ks & 1][x - 1] = read_a(st, std::integral_constant<int, x - 1>{}, ks_tag);
                else fb[ks & 1][1] = read_b(st, std::integral_constant<int, 1>{}, ks_tag);
            };
            auto multiply = [&](auto m_tag, auto ks_tag) __attribute__((always_inline)) {
                constexpr int m = decltype(m_tag)::value, ks = decltype(ks_tag)::value, j = m / L, i = m % L;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[i][j], 0, 0, 0);
            };
            bf_static_for<0, NR>([&](auto x) { read(x, std::integral_constant<int, 0>{}, smem); });
            for (int s = 0; s < nfull; ++s) {
                uint8_t* cur = smem + (s & 1) * TL_STAGE;
                uint8_t* nxt = smem + ((s & 1) ^ 1) * TL_STAGE;
                bf_static_for<0, 3>([&](auto ks_tag) {
                    constexpr int ks = decltype(ks_tag)::value;
                    bf_static_for<0, NM>([&](auto m_tag) {
                        constexpr int m = decltype(m_tag)::value;
                        multiply(m_tag, ks_tag);
                        bf_static_for<(m * NR + NM - 1) / NM, ((m + 1) * NR + NM - 1) / NM>([&](auto x) { read(x, std::integral_constant<int, ks + 1>{}, cur); });
                        if constexpr (ks < 1) {
                            constexpr int q = (NM - NB) + ks * NM + m;
                            bf_static_for<q * TL_REQ / Q, (q + 1) * TL_REQ / Q>([&](auto e) { request(e, in, tl); });
                        }
                        if constexpr (ks == 1 && m == 1) ask_l2(tl, s + TL_AHEAD);
                        __builtin_amdgcn_sched_barrier(0);
                    });
                });
                bf_static_for<0, NB>([&](auto m_tag) { multiply(m_tag, std::integral_constant<int, 3>{}); });
                in = in_begin(tl, s + 2);
                bf_wait_vm<1>();        // slot s + 1 has landed (the L2 request may still be on its way)
                __syncthreads();        // ... for every wave, and every wave holds its fragments of slot s
                __builtin_amdgcn_sched_barrier(0);
                bf_static_for<NB, NM>([&](auto m_tag) {
                    constexpr int m = decltype(m_tag)::value, q = m - NB;
                    multiply(m_tag, std::integral_constant<int, 3>{});
                    bf_static_for<(q * NR + NM - NB - 1) / (NM - NB), ((q + 1) * NR + NM - NB - 1) / (NM - NB)>([&](auto x) { read(x, std::integral_constant<int, 0>{}, nxt); });
                    bf_static_for<q * TL_REQ / Q, (q + 1) * TL_REQ / Q>([&](auto e) { request(e, in, tl); });
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
            if (halves & 1) {           // the last slot's first half
                uint8_t* cur = smem + (nfull & 1) * TL_STAGE;
                bf_static_for<0, NR>([&](auto x) { read(x, std::integral_constant<int, 1>{}, cur); });
                bf_static_for<0, 2>([&](auto ks_tag) { bf_static_for<0, NM>([&](auto m_tag) { multiply(m_tag, ks_tag); }); });
            }
        };
        if (halves > 0) {
            if (live > 2) run(std::integral_constant<int, 4>{});
            else if (live > 0) run(std::integral_constant<int, 2>{});
            else {
                // no row or column of the tile is this wave's: it only keeps its share of the requests going
                In in = in_begin(tl, 1);
                bf_static_for<0, TL_REQ>([&](auto e) { request(e, in, tl); });
                bf_wait_vm<TL_REQ>();
                __syncthreads();
                for (int s = 0; s < nfull; ++s) {
                    ask_l2(tl, s + TL_AHEAD);
                    bf_wait_vm<1>();
                    __syncthreads();
                    in = in_begin(tl, s + 2);
                    bf_static_for<0, TL_REQ>([&](auto e) { request(e, in, tl); });
                }
            }
        }
        bf_wait_vm<0>();
        __syncthreads();         // every wave is done with the stages

        // the next tile's first slot goes into stage 0 while this tile's output leaves through stage 1
        const int grp = tl.grp, m_valid = tl.m_valid, n_valid = tl.n_valid;
        const int64_t n0 = tl.n0, c_row0 = tl.c_row0;
        tile_id += nwg;
        const bool more = tile_id < total_tiles;
        if (more) {
            tl = setup(tile_id);
            first_slot(tl);
        }

        // lane (lr, g) of fragment (i, j) holds row 32 i + lr, columns 32 j + 8 q + 4 g .. + 3 in registers 4 q .. 4 q + 3
        if (ACCUM) {
            float* c = (float*)p.c + ((int64_t)grp * p.m + c_row0) * p.n + n0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wm * 128 + 32 * i + lr;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int col = wn * 64 + 32 * j + 8 * q + 4 * g;
                        if (row < m_valid && col < n_valid) {      // n_out is a multiple of 8: a quad is in or out as a whole
                            v4f* dst = (v4f*)(c + (int64_t)row * p.n + col);
                            v4f o = *dst;
                            o[0] += acc[i][j][4 * q]; o[1] += acc[i][j][4 * q + 1]; o[2] += acc[i][j][4 * q + 2]; o[3] += acc[i][j][4 * q + 3];
                            *dst = o;
                        }
                    }
            }
        } else {
            uint16_t* c = (uint16_t*)p.c + ((WGRAD ? (int64_t)grp * p.m : 0) + c_row0) * p.n + n0;
            // in two passes of 128 rows of 512 bytes, 16-byte pieces XOR row % 32; every wave stores whole rows
            uint8_t* out = smem + TL_STAGE;
            int to = t;
            asm("" : "+v"(to));          // the store addresses are formed here, not kept in registers across the main loop
            const int col = (to & 31) * 8, row0 = to >> 5;
            // Non-temporal stores through a descriptor that ends with the tile's last row, columns past the last one sent
            // past every end: no branch around a store, and the L2 is left to the operands.  32 groups of about 1024 rows,
            // [4096, 7168], forward / dgrad / weight gradient 1820 / 1714 / 1731 -> 1810 / 1696 / 1703 us, [7168, 2048]
            // 904 / 901 / 895 -> 890 / 897 / 881.  (Letting them be on their way in the next tile's first slot: +- 0.)
            const uint32_t row_bytes = (uint32_t)p.n * 2;
            const uint32_t at = col < n_valid ? (uint32_t)row0 * row_bytes + (uint32_t)col * 2 : addr::kDropped;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (h) __syncthreads();
                if (wm == h) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const v4bf o = {(__bf16)acc[i][j][4 * q], (__bf16)acc[i][j][4 * q + 1], (__bf16)acc[i][j][4 * q + 2], (__bf16)acc[i][j][4 * q + 3]};
                                *(v4bf*)(out + (32 * i + lr) * 512 + 16 * ((8 * wn + 4 * j + q) ^ lr) + 8 * g) = o;
                            }
                }
                __syncthreads();
                uint4 v[8];
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    const int row = x * 16 + row0;
                    v[x] = *(const uint4*)(out + row * 512 + 16 * ((to & 31) ^ (row & 31)));
                }
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    const int row = h * 128 + x * 16;
                    const int rows = m_valid - row;
                    const auto rs = __builtin_amdgcn_make_buffer_rsrc(c + (int64_t)row * p.n, 0, rows > 0 ? (rows < 16 ? rows : 16) * (int)row_bytes : 0, 0x00020000);
                    const u32x4 o = {v[x].x, v[x].y, v[x].z, v[x].w};
                    constexpr int kNonTemporal = 2;
                    __builtin_amdgcn_raw_buffer_store_b128(o, rs, (int)at, 0, kNonTemporal);
                }
            }
        }
        if (!more) break;
        __syncthreads();         // every wave has left the staging area: the next tile's requests may overwrite it
    }
}

static int bf16_num_cus(int dev) {
    static std::atomic<int> cached[64];
    int v = cached[dev & 63].load(std::memory_order_relaxed);
    if (v) return v;
    hipDeviceProp_t pr;
    if (hipGetDeviceProperties(&pr, dev) != hipSuccess || pr.multiProcessorCount <= 0) return 256;
    cached[dev & 63].store(pr.multiProcessorCount, std::memory_order_relaxed);
    return pr.multiProcessorCount;
}

template <int BM, bool A_T, bool B_T, bool WGRAD, bool ACCUM>
static int launch_bf16(const Bf16Args& a, int64_t max_tiles, hipStream_t st) {
    constexpr bool TALL = BM == 256;
    constexpr int lds = TALL ? tall_lds_bytes() : bf16_lds_bytes();
    if (!device_is_gfx950()) return MXL_ENODEV;
    static std::atomic<bool> attr_set[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return MXL_ELAUNCH;
    void (*kern)(Bf16Args) = nullptr;
    if constexpr (TALL) kern = bf16_gemm_tall_kernel<A_T, B_T, WGRAD, ACCUM>;
    else kern = bf16_gemm_kernel<A_T, B_T, WGRAD, ACCUM>;
    if (!attr_set[dev & 63].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return MXL_ELAUNCH;
        attr_set[dev & 63].store(true, std::memory_order_release);
    }
    if (max_tiles <= 0) return MXL_OK;
    if (max_tiles > 0x7FFFFFFF) return MXL_EINVAL;
    // persistent: as many workgroups as the device holds at once (a multiple of 8, one share per XCD), fewer for few tiles
    int64_t grid = (int64_t)bf16_num_cus(dev) * (BM == 256 ? 1 : 2);
    grid = grid / 8 * 8;
    if (grid < 8) grid = 8;
    if ((max_tiles + 7) / 8 * 8 < grid) grid = (max_tiles + 7) / 8 * 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(TALL ? TL_THREADS : BF_THREADS), lds, st, a);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

// Tile height of a launch: the caller's choice (MXL_BF_TILE_128 / MXL_BF_TILE_256), else from the average number of
// rows per group -- the counts live on the device, the average is all the host knows.  Forward / dgrad tiles are cut from
// a group's rows, and 256-row tiles win from about 256 rows per group on (32 groups, [4096, 7168], forward + dgrad with
// 256-row against 128-row tiles: 1024 rows 3.42 against 4.16 ms, 256 rows 1.49 against 1.55, 128 rows 1.23 against 1.16).
// The weight gradient's are cut from the output: 256 rows are as fast or faster at every length (1024 rows 1.71 against
// 1.94 ms, 256 rows 0.72 against 0.78, 64 rows 0.43 against 0.44).
static bool bf16_tall_tiles(uint32_t flags, int64_t rows_per_group, int64_t threshold) {
    if (flags & MXL_BF_TILE_256) return true;
    if (flags & MXL_BF_TILE_128) return false;
    return rows_per_group >= threshold;
}

}  // namespace mxl

using namespace mxl;

extern "C" int mxl_grouped_gemm_bf16(const void* a_bf16, const void* b_bf16, void* c_bf16, const int64_t* group_lens,
                                     int num_groups, int64_t total_m, int64_t n, int64_t k, uint32_t flags, void* stream) {
    if (flags & ~(uint32_t)(MXL_BF_B_KN | MXL_BF_TILE_128 | MXL_BF_TILE_256)) return MXL_EINVAL;
    if ((flags & MXL_BF_TILE_128) && (flags & MXL_BF_TILE_256)) return MXL_EINVAL;
    if (total_m < 0 || n <= 0 || k <= 0 || n % 8 != 0 || k % BF_KS != 0) return MXL_EINVAL;
    if (num_groups < 1 || num_groups > MXL_MAX_GROUPS || (num_groups > 1 && !group_lens)) return MXL_EINVAL;
    if (total_m == 0) return MXL_OK;
    if (!a_bf16 || !b_bf16 || !c_bf16) return MXL_EINVAL;
    if ((((uintptr_t)a_bf16 | (uintptr_t)b_bf16 | (uintptr_t)c_bf16) & 15) != 0) return MXL_EINVAL;
    // offsets inside a tile's operand rows are 32-bit
    if (256 * k * 2 >= ((int64_t)1 << 31) || k * n * 2 >= ((int64_t)1 << 32)) return MXL_EINVAL;
    Bf16Args a{(const uint8_t*)a_bf16, (const uint8_t*)b_bf16, c_bf16, group_lens, num_groups, total_m, 0, n, k};
    const bool tall = bf16_tall_tiles(flags, total_m / num_groups, 256);
    const int64_t max_tiles = (total_m / (tall ? 256 : 128) + num_groups) * ((n + BF_BN - 1) / BF_BN);
    hipStream_t st = (hipStream_t)stream;
    if (flags & MXL_BF_B_KN)
        return tall ? launch_bf16<256, false, true, false, false>(a, max_tiles, st) : launch_bf16<128, false, true, false, false>(a, max_tiles, st);
    return tall ? launch_bf16<256, false, false, false, false>(a, max_tiles, st) : launch_bf16<128, false, false, false, false>(a, max_tiles, st);
}

extern "C" int mxl_grouped_gemm_bf16_wgrad(const void* p_bf16, const void* q_bf16, void* c, const int64_t* group_lens,
                                           int num_groups, int64_t total_m, int64_t m_out, int64_t n_out, uint32_t flags,
                                           void* stream) {
    if (flags & ~(uint32_t)(MXL_BF_ACCUM_F32 | MXL_BF_TILE_128 | MXL_BF_TILE_256)) return MXL_EINVAL;
    if ((flags & MXL_BF_TILE_128) && (flags & MXL_BF_TILE_256)) return MXL_EINVAL;
    if (total_m < 0 || m_out <= 0 || n_out <= 0 || m_out % 8 != 0 || n_out % 8 != 0) return MXL_EINVAL;
    if (num_groups < 1 || num_groups > MXL_MAX_GROUPS || (num_groups > 1 && !group_lens)) return MXL_EINVAL;
    if (!c || ((uintptr_t)c & 15) != 0) return MXL_EINVAL;
    if (total_m > 0 && (!p_bf16 || !q_bf16 || (((uintptr_t)p_bf16 | (uintptr_t)q_bf16) & 15) != 0)) return MXL_EINVAL;
    // the K-slot advance inside a group's token range is a 32-bit byte offset
    if (total_m * m_out * 2 >= ((int64_t)1 << 32) || total_m * n_out * 2 >= ((int64_t)1 << 32)) return MXL_EINVAL;
    Bf16Args a{(const uint8_t*)p_bf16, (const uint8_t*)q_bf16, c, group_lens, num_groups, total_m, m_out, n_out, 0};
    // the tiles are cut from the [m_out, n_out] matrix of every group; the contraction runs over the group's tokens
    // (the last K slot may reach 63 tokens past the operand's end, where 32-bit offsets must not wrap around)
    const bool tall = bf16_tall_tiles(flags, total_m / num_groups, 0) && (total_m + 64) * (m_out > n_out ? m_out : n_out) * 2 < ((int64_t)1 << 32);
    const int bm = tall ? 256 : 128;
    const int64_t max_tiles = (int64_t)num_groups * ((m_out + bm - 1) / bm) * ((n_out + BF_BN - 1) / BF_BN);
    hipStream_t st = (hipStream_t)stream;
    if (flags & MXL_BF_ACCUM_F32)
        return tall ? launch_bf16<256, true, true, true, true>(a, max_tiles, st) : launch_bf16<128, true, true, true, true>(a, max_tiles, st);
    return tall ? launch_bf16<256, true, true, true, false>(a, max_tiles, st) : launch_bf16<128, true, true, true, false>(a, max_tiles, st);
}
