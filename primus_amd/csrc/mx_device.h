// Device-side helpers shared by the MX quantisers and GEMMs (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mxlinear.h"

#include <string.h>

#include <atomic>

namespace mxl {

// Host side: is the current device a gfx950?  The kernels exist for that target only; every entry point
// asks before its first launch on a device (answer cached per device index) and returns MXL_ENODEV otherwise.
inline bool device_is_gfx950() {
    static std::atomic<int> known[64];   // 0 unknown, 1 yes, 2 no
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    const int slot = dev & 63;
    int v = known[slot].load(std::memory_order_relaxed);
    if (v == 0) {
        hipDeviceProp_t pr;
        if (hipGetDeviceProperties(&pr, dev) != hipSuccess) return false;
        v = strncmp(pr.gcnArchName, "gfx950", 6) == 0 ? 1 : 2;
        known[slot].store(v, std::memory_order_relaxed);
    }
    return v == 1;
}

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

constexpr int kFmtE4M3 = MXL_FMT_E4M3;
constexpr int kFmtE2M1 = MXL_FMT_E2M1;
constexpr int kFmtE5M2 = MXL_FMT_E5M2;   // tensor-wise scaled operands only (gradients of the HYBRID format)

// Exponent of the largest normal, its fp32 mantissa field, explicit mantissa bits.
template <int FMT> struct Elem;
template <> struct Elem<kFmtE4M3> {
    static constexpr int emax = 8;
    static constexpr uint32_t maxman = 0x600000u;  // 448 = 1.75 * 2^8
    static constexpr int mbits = 3;
};
template <> struct Elem<kFmtE2M1> {
    static constexpr int emax = 2;
    static constexpr uint32_t maxman = 0x400000u;  // 6 = 1.5 * 2^2
    static constexpr int mbits = 1;
};

// E8M0 byte of a block from the largest bf16 magnitude in it (15-bit pattern).
// Integer arithmetic on the fp32 exponent field only; 255 marks a block that
// holds a NaN or an infinity.
template <int FMT, int SMODE>
__device__ __forceinline__ uint32_t scale_byte(uint32_t amax16) {
    uint32_t b = amax16 << 16;
    if (SMODE == MXL_SCALE_EVEN) b += 1u << (23 - Elem<FMT>::mbits - 1);
    int e = (int)(b >> 23);
    if (SMODE == MXL_SCALE_RCEIL) e += ((b & 0x7FFFFFu) > Elem<FMT>::maxman) ? 1 : 0;
    e -= Elem<FMT>::emax;
    e = e < 0 ? 0 : (e > 254 ? 254 : e);
    return amax16 >= 0x7F80u ? 255u : (uint32_t)e;
}

// 2^(127 - byte) for byte <= 253 (always a normal float).
__device__ __forceinline__ float inv_scale(uint32_t byte) { return __uint_as_float((254u - byte) << 23); }
// 2^(byte - 127) for byte in [1, 254]; byte 0 gives the subnormal 2^-127.
__device__ __forceinline__ float fwd_scale(uint32_t byte) {
    return byte ? __uint_as_float(byte << 23) : __uint_as_float(0x00400000u);
}

__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xFFFF0000u); }

// Largest magnitude (as 15-bit patterns) of the two bf16 halves, lane-wise packed.
__device__ __forceinline__ uint32_t pk_absmax(uint32_t acc, uint32_t pair) {
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    us2 a = __builtin_bit_cast(us2, acc);
    us2 b = __builtin_bit_cast(us2, pair & 0x7FFF7FFFu);
    us2 r = {(unsigned short)(a[0] > b[0] ? a[0] : b[0]), (unsigned short)(a[1] > b[1] ? a[1] : b[1])};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t pk_max16(uint32_t x, uint32_t y) {
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    us2 a = __builtin_bit_cast(us2, x);
    us2 b = __builtin_bit_cast(us2, y);
    us2 r = {(unsigned short)(a[0] > b[0] ? a[0] : b[0]), (unsigned short)(a[1] > b[1] ? a[1] : b[1])};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t hmax16(uint32_t pk) {
    uint32_t lo = pk & 0xFFFFu, hi = pk >> 16;
    return lo > hi ? lo : hi;
}

// Two bf16 (packed) -> two E4M3 bytes in the low 16 bits.  `inv` is the
// power-of-two factor; the clamp makes the hardware convert (round to nearest
// even, NaN on overflow) saturating.
__device__ __forceinline__ uint32_t cvt2_e4m3(uint32_t pair, float inv) {
    float a = __builtin_amdgcn_fmed3f(bf16_lo(pair) * inv, -448.f, 448.f);
    float b = __builtin_amdgcn_fmed3f(bf16_hi(pair) * inv, -448.f, 448.f);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xFFFFu;
}
// Four bf16 (two packed pairs) -> four E4M3 bytes.
__device__ __forceinline__ uint32_t cvt4_e4m3(uint32_t p0, uint32_t p1, float inv) {
    float a = __builtin_amdgcn_fmed3f(bf16_lo(p0) * inv, -448.f, 448.f);
    float b = __builtin_amdgcn_fmed3f(bf16_hi(p0) * inv, -448.f, 448.f);
    float c = __builtin_amdgcn_fmed3f(bf16_lo(p1) * inv, -448.f, 448.f);
    float d = __builtin_amdgcn_fmed3f(bf16_hi(p1) * inv, -448.f, 448.f);
    int r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
    return (uint32_t)r;
}
// The same for E5M2 (tensor-wise scaled gradients): multiply, clamp at +-57344, round to nearest even.
__device__ __forceinline__ uint32_t cvt4_e5m2(uint32_t p0, uint32_t p1, float inv) {
    float a = __builtin_amdgcn_fmed3f(bf16_lo(p0) * inv, -57344.f, 57344.f);
    float b = __builtin_amdgcn_fmed3f(bf16_hi(p0) * inv, -57344.f, 57344.f);
    float c = __builtin_amdgcn_fmed3f(bf16_lo(p1) * inv, -57344.f, 57344.f);
    float d = __builtin_amdgcn_fmed3f(bf16_hi(p1) * inv, -57344.f, 57344.f);
    int r = __builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_bf8_f32(c, d, r, true);
    return (uint32_t)r;
}
template <int FMT> __device__ __forceinline__ uint32_t cvt4_fp8(uint32_t p0, uint32_t p1, float inv) {
    return FMT == kFmtE5M2 ? cvt4_e5m2(p0, p1, inv) : cvt4_e4m3(p0, p1, inv);
}
// Slow path for a block that holds a NaN/Inf: finite lanes -> signed zero,
// non-finite lanes -> NaN code with the input's sign.
__device__ __forceinline__ uint32_t nonfinite1_e4m3(uint32_t h) {
    uint32_t s = (h >> 8) & 0x80u;
    return ((h & 0x7FFFu) >= 0x7F80u) ? (s | 0x7Fu) : s;
}
__device__ __forceinline__ uint32_t nonfinite4_e4m3(uint32_t p0, uint32_t p1) {
    return nonfinite1_e4m3(p0 & 0xFFFFu) | (nonfinite1_e4m3(p0 >> 16) << 8) | (nonfinite1_e4m3(p1 & 0xFFFFu) << 16) |
           (nonfinite1_e4m3(p1 >> 16) << 24);
}

// Two bf16 (packed) -> two E2M1 nibbles in bits 7:0 (element 0 in bits 3:0).
// The hardware convert divides by `scale` (a power of two), rounds to nearest
// even and saturates at +-6.
__device__ __forceinline__ uint32_t cvt2_e2m1(uint32_t pair, float scale) {
    v2bf h = __builtin_bit_cast(v2bf, pair);
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(0u, h, scale, 0) & 0xFFu;
}
__device__ __forceinline__ uint32_t nonfinite1_e2m1(uint32_t h) {
    uint32_t s = (h >> 12) & 0x8u;
    return ((h & 0x7FFFu) >= 0x7F80u) ? (s | 0x7u) : s;
}
__device__ __forceinline__ uint32_t nonfinite2_e2m1(uint32_t pair) {
    return nonfinite1_e2m1(pair & 0xFFFFu) | (nonfinite1_e2m1(pair >> 16) << 4);
}

// ---- stochastic rounding to E2M1 (gradients of the MXFP4 recipe: rowwise_use_sr / colwise_use_sr of
// quantize_mxfp4_dual, primus/backends/megatron/core/extensions/primus_turbo_mxfp4_local.py:272-288).
// Integer arithmetic throughout so that a CPU restatement reproduces every code:
//   w = |x| * 2^(127 - scale byte)                         (exact: power-of-two scaling of a bf16)
//   w >= 1: the fp32 pattern of w plus a random integer below 2^22, cut after one mantissa bit
//           (round up with probability = the dropped fraction), saturating at 6;
//   w <  1: floor(w * 2^23) plus the same random integer, cut at 2^22  -> 0, 0.5 or 1.
// Random bits: a counter-based hash, 16 bits per element, two elements per 32-bit word.
__device__ __forceinline__ uint32_t sr_mix(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7FEB352Du;
    x ^= x >> 15;
    x *= 0x846CA68Bu;
    x ^= x >> 16;
    return x;
}
// The word of counter `key + i`, i < 4, key a multiple of 4: `low` = key's low word ^ the seed's, `high` = sr_high(), the
// part that the four words of a key share.
__device__ __forceinline__ uint32_t sr_high(uint64_t key, uint64_t seed, uint32_t stream) {
    return (uint32_t)(key >> 32) * 0x9E3779B9u + (uint32_t)(seed >> 32) + stream * 0x85EBCA6Bu;
}
__device__ __forceinline__ uint32_t sr_word(uint32_t low, uint32_t i, uint32_t high) { return sr_mix(sr_mix(low ^ i) + high); }
// (The products of the counter and the shared part are worked out once.  The kernel is bound by instructions, 148 for eight codes:
// quantising [4096, 14336] both ways with stochastic rounding and the Hadamard transform takes 87 us, 46 without stochastic rounding; 91
// with a conversion to integers and a median per magnitude and the nibbles put together one by one, 163 instructions.  The four
// words' first products out of one multiplication are 8 additions for 3 multiplications: 89.5; products out of 16-bit dot products: 101.)
// The magnitude without a branch, in bits 26:24 of the result (the caller takes the upper byte).  In units of 2^-23 it is w below 1
// and w's fp32 pattern, less that of 0.5, from 1 on.  The first comes out of the pattern of (w + 1) 2^23 - 0.5, less that of 2^23 and
// not below it.  The sum may round to the integer below, but never across a multiple of 64 (w has 8 bits: 63.25 to 63.75 and 127.5
// stay below, 64 and 128 do not), and what is added is a multiple of 64.  The larger of the two is the one wanted: below 1 the pattern of w is
// the smaller, from 1 on that of w + 1 is.  Both carry the pattern of 2^23 here, which the random bits' upper byte takes off again.
constexpr uint32_t SR_RND_TOP = 0xD4000000u;      // -(0x4B000000 << 2)
__device__ __forceinline__ uint32_t sr_mag_e2m1(float x, float inv, uint32_t rnd8) {
    const float w = fabsf(x) * inv;
    const uint32_t fixed = __float_as_uint(fmaf(w, 8388608.f, 8388607.5f)), line = __float_as_uint(w) + (0x4B000000u - 0x3F000000u);
    return min((max(max(fixed, line), 0x4B000000u) << 2) + rnd8, 0x7FFFFFFu);
}
// four packed bf16 pairs -> eight nibbles, element 0 (random bits 15:0 of the first word) in bits 3:0; the signs are
// gathered for all eight at once.  key: the first pair's counter, a multiple of 4
__device__ __forceinline__ uint32_t sr8_e2m1(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3, float inv, uint64_t key,
                                             uint64_t seed, uint32_t stream) {
    const uint32_t p[4] = {p0, p1, p2, p3};
    const uint32_t low = (uint32_t)key ^ (uint32_t)seed, high = sr_high(key, seed, stream);
    uint32_t e[4], d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t rnd = sr_word(low, (uint32_t)i, high);
        e[i] = sr_mag_e2m1(bf16_lo(p[i]), inv, __builtin_amdgcn_perm(SR_RND_TOP, rnd, 0x0701000Cu));      // bits 15:0, from bit 8 on
        d[i] = sr_mag_e2m1(bf16_hi(p[i]), inv, __builtin_amdgcn_perm(SR_RND_TOP, rnd, 0x0703020Cu));      // bits 31:16
    }
    const uint32_t e_all = __builtin_amdgcn_perm(__builtin_amdgcn_perm(e[3], e[2], 0x07030C0Cu), __builtin_amdgcn_perm(e[1], e[0], 0x0C0C0703u), 0x07060100u);
    const uint32_t d_all = __builtin_amdgcn_perm(__builtin_amdgcn_perm(d[3], d[2], 0x07030C0Cu), __builtin_amdgcn_perm(d[1], d[0], 0x0C0C0703u), 0x07060100u);
    const uint32_t o = e_all | (d_all << 4);
    const uint32_t x = __builtin_amdgcn_perm(p1, p0, 0x07030501u), y = __builtin_amdgcn_perm(p3, p2, 0x07030501u);
    const uint32_t even = __builtin_amdgcn_perm(y, x, 0x05040100u), odd = __builtin_amdgcn_perm(y, x, 0x07060302u);
    return o | ((even >> 4) & 0x08080808u) | (odd & 0x80808080u);
}

// ---- gated activation of the expert MLP (shared by the activation kernels and the fused
// activation + quantisation path, so that both round identically) ----
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    v2bf h = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, h);
}
template <int ACT> __device__ __forceinline__ float act_fwd(float g) {
    // hardware exp2 and reciprocal (about 1 ulp each in fp32, far inside the bf16 rounding of the result); the
    // IEEE division and the range handling of expf would make the fused quantiser ALU-bound
    if (ACT == MXL_ACT_SILU) return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
    // 0.5 g erfc(-g / sqrt 2); erfc (not 1 + erf): no cancellation in the negative tail.  erfc(z), z >= 0, from
    // the rational-exponential fit t exp(-z^2 + P(t)), t = 1 / (1 + z / 2) (fractional error below 1.2e-7
    // everywhere, Numerical Recipes 6.2), with the hardware reciprocal and exp2: the library erfcf would make
    // the fused quantiser ALU-bound.
    const float x = g * -0.70710678118654752f, z = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(1.f + 0.5f * z);
    float p = 0.17087277f;
    p = p * t - 0.82215223f;
    p = p * t + 1.48851587f;
    p = p * t - 1.13520398f;
    p = p * t + 0.27886807f;
    p = p * t - 0.18628806f;
    p = p * t + 0.09678418f;
    p = p * t + 0.37409196f;
    p = p * t + 1.00002368f;
    p = p * t - 1.26551223f;
    const float e = t * __builtin_amdgcn_exp2f((p - z * z) * 1.4426950408889634f);
    return 0.5f * g * (x >= 0.f ? e : 2.f - e);
}
__device__ __forceinline__ float load_prob(const void* probs, int probs_bf16, int64_t row) {
    if (probs_bf16) return __uint_as_float((uint32_t)((const uint16_t*)probs)[row] << 16);
    return ((const float*)probs)[row];
}
// 8 outputs act(g) * u * p from 8 gate and 8 linear bf16 values, rounded once to bf16
template <int ACT> __device__ __forceinline__ uint4 glu8(const uint4& g, const uint4& u, float p) {
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    uint32_t ow[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float lo = act_fwd<ACT>(bf16_lo(gw[k])) * bf16_lo(uw[k]) * p;
        const float hi = act_fwd<ACT>(bf16_hi(gw[k])) * bf16_hi(uw[k]) * p;
        ow[k] = pack_bf16(lo, hi);
    }
    return make_uint4(ow[0], ow[1], ow[2], ow[3]);
}

// ---- RMSNorm (shared by the normalisation kernels and the fused normalisation + quantisation path) ----
// 8 outputs (x * rstd) * w from 8 input and 8 weight bf16 values, fp32 products in that order, rounded once
__device__ __forceinline__ uint4 norm8(const uint4& x, const uint4& wv, float rstd) {
    const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, ww[4] = {wv.x, wv.y, wv.z, wv.w};
    uint32_t ow[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        ow[k] = pack_bf16(bf16_lo(xw[k]) * rstd * bf16_lo(ww[k]), bf16_hi(xw[k]) * rstd * bf16_hi(ww[k]));
    return make_uint4(ow[0], ow[1], ow[2], ow[3]);
}

// ---- shared by the quantisers ----
// The quantisers stream: every input byte is read once and every output byte written once, by one
// workgroup.  Non-temporal accesses keep that traffic from displacing the scale words in L2, which
// do have to wait there for their neighbours (the 8 x 8 supertile order of the quantisers' grids).
typedef uint32_t qu32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t qu32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store16_streaming(void* d, const uint4& v) {
    const qu32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, (qu32x4*)d);
}
__device__ __forceinline__ void store8_streaming(void* d, const uint2& v) {
    const qu32x2 t = {v.x, v.y};
    __builtin_nontemporal_store(t, (qu32x2*)d);
}
__device__ __forceinline__ void store4_streaming(void* d, uint32_t v) { __builtin_nontemporal_store(v, (uint32_t*)d); }
// Through the caches (`keep`) or past them.  The empty statements keep the compiler from making one store of the two, which would
// not be a streaming one.
__device__ __forceinline__ void store16(void* d, const uint4& v, bool keep) {
    if (keep) {
        asm volatile("");
        *(uint4*)d = v;
        asm volatile("");
    } else {
        store16_streaming(d, v);
    }
}
__device__ __forceinline__ void store4(void* d, uint32_t v, bool keep) {
    if (keep) {
        asm volatile("");
        *(uint32_t*)d = v;
        asm volatile("");
    } else {
        store4_streaming(d, v);
    }
}
__device__ __forceinline__ uint4 load16_streaming(const void* s) {
    const qu32x4 t = __builtin_nontemporal_load((const qu32x4*)s);
    return make_uint4(t.x, t.y, t.z, t.w);
}

__device__ __forceinline__ uint32_t dpp_xor1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ uint32_t dpp_xor2(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
}
// the other two steps of a maximum over the 16 lanes of a DPP row: lane i <-> 7 - i inside each half row, lane i <-> 15 - i
__device__ __forceinline__ uint32_t dpp_half_mirror(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true);  // row_half_mirror
}
__device__ __forceinline__ uint32_t dpp_mirror(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true);  // row_mirror
}


// ---- ragged groups ----
// Inclusive prefix sum over the wave's 64 lanes, saturating at 2^32 - 1: six additions with DPP operands (row_shr 1, 2, 4, 8,
// row_bcast 15 and 31).
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false));
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false));
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false));
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false));
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));
    v = __builtin_elementwise_add_sat(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));
    return v;
}

// The groups' lens summed up by one wave, 64 groups at a time: step(lens, c) gives lane l of group c + l the elements in front
// of the group and with it.  Lens are clamped to what the operand holds (`cap` < 2^32 - 127: negative ones read as 0, the running
// sum never passes cap), so that lens which do not match the buffers cannot send a tile outside them; with ALIGN each is
// rounded up first.  Against one thread that adds the lens up one after the other, a load or an LDS access each, us: both
// copies of [512, 1024] in 32, 128, 256 groups 10.6, 38, 104 -> 7.4, 14, 23 (every workgroup of the quantiser does it); the ring
// kernel on [1024, 1024] weights, 512 rows, 16.8, 42, 78 -> 13.9, 32, 60.
template <uint32_t ALIGN = 1> struct GroupScan {
    uint32_t cap, base = 0;
    int groups, lane;
    __device__ __forceinline__ GroupScan(int64_t cap_, int groups_, int lane_) : cap((uint32_t)cap_), groups(groups_), lane(lane_) {}
    // lens null: one group that has everything
    __device__ __forceinline__ void step(const int64_t* lens, int c, uint32_t& first, uint32_t& end) {
        const int i = c + lane;
        int64_t len = i < groups ? (lens ? lens[i] : (int64_t)cap) : 0;
        len = len < 0 ? 0 : len > (int64_t)cap ? (int64_t)cap : len;
        uint32_t v = ((uint32_t)len + (ALIGN - 1)) / ALIGN * ALIGN;
        v = v < cap ? v : cap;
        end = __builtin_elementwise_add_sat(wave_prefix(v), base);
        end = end < cap ? end : cap;
        first = (uint32_t)__builtin_amdgcn_update_dpp((int)base, (int)end, 0x138, 0xF, 0xF, false);   // wave_shr 1
        base = (uint32_t)__builtin_amdgcn_readlane((int)end, 63);
    }
};

}  // namespace mxl
