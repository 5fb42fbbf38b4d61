// Gated activation of the expert MLP fused with the router probability and the row mask
// (swiglu_with_probs / geglu_with_probs as called by the reference's fused_bias_act_with_probs,
// primus/backends/megatron/core/extensions/primus_turbo.py:1954-1980; unfused arithmetic at
// primus/backends/megatron/core/transformer/experts.py:100-118):
//
//   y[m, j] = act(x[m, j]) * x[m, F + j] * p[m]            rows with mask 0 give 0
//
// for bf16 x[rows, 2F], computed in fp32 and rounded once to bf16.  Backward returns dx[rows, 2F]
// and dp[rows] (fp32).  Both kernels stream: one workgroup per row, 16 bytes per lane and access.
//
// Bound by memory (6 and 10 bytes per output element), at 6.0-6.4 TB/s where a workgroup gets through its row in one to two
// passes: with 256 threads a long row is many short visits to each of its pieces of memory while thousands of others are open.
// Hence 256, 512 or 1024 threads by the row's length.  us, 256 / 512 / 1024 threads: backward [32768, 14336] 882 / 846 / 813,
// [8192, 14336] 219 / 208 / 194, [8192, 7168] 105 / 98 / 95, [8192, 5760] 83 / 77 / 83, [16384, 3584] 97 / 91 / 117, [65536, 2880]
// 311 / 306 / 408, [32768, 2048] 106 / 114 / 172; forward 506 / 481 / 461, 127 / 116 / 111, 60 / 56 / 57, 47 / 45 / 47, 55 / 57 / 59,
// 176 / 175 / 188, 64 / 64 / 64.
#include "mx_activation.h"
#include "mx_device.h"

namespace mxl {

constexpr int ATHREADS = 256;     // (row_mask_kernel)

typedef uint32_t au32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 act_load16(const void* s) {
    const au32x4 t = __builtin_nontemporal_load((const au32x4*)s);
    return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ void act_store16(void* d, const uint4& v) {
    const au32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, (au32x4*)d);
}
// act(g) together with its derivative, fp32
template <int ACT> __device__ __forceinline__ void act_both(float g, float& a, float& da) {
    if (ACT == MXL_ACT_SILU) {
        const float s = 1.f / (1.f + expf(-g));
        a = g * s;
        da = s * (1.f + g * (1.f - s));
    } else {
        const float c = 0.5f * erfcf(-g * 0.70710678118654752f);
        a = g * c;
        da = c + g * 0.39894228040143268f * expf(-0.5f * g * g);
    }
}

template <int ACT, int THREADS>
__global__ __launch_bounds__(THREADS) void glu_probs_fwd_kernel(const uint16_t* x, const void* probs, int probs_bf16,
                                                                 const uint8_t* row_mask, int64_t f, uint16_t* y) {
    const int64_t row = blockIdx.x;
    const bool live = row_mask == nullptr || row_mask[row] != 0;
    const float p = live ? load_prob(probs, probs_bf16, row) : 0.f;
    const uint16_t* xg = x + row * 2 * f;
    uint16_t* yr = y + row * f;
    for (int64_t c = (int64_t)threadIdx.x * 8; c < f; c += THREADS * 8) {
        uint4 o = make_uint4(0, 0, 0, 0);
        if (live) {
            o = glu8<ACT>(act_load16(xg + c), act_load16(xg + f + c), p);
        }
        act_store16(yr + c, o);
    }
}

// SUMS: partial sums a thread keeps.  The gradient of a row's probability is a sum over the row whose order is that of THREADS * SUMS
// threads with one sum each: chunk i of a thread goes to sum i mod SUMS, which is what thread threadIdx.x + THREADS * (i mod SUMS) of
// those has, and the waves' sums are added in their order.  So a smaller workgroup gives the bits of the one it stands in for.
template <int ACT, int THREADS, int SUMS>
__global__ __launch_bounds__(THREADS) void glu_probs_bwd_kernel(const uint16_t* dy, const uint16_t* x, const void* probs,
                                                                 int probs_bf16, const uint8_t* row_mask, int64_t f,
                                                                 uint16_t* dx, float* dprobs) {
    __shared__ float part[SUMS * THREADS / 64];
    const int64_t row = blockIdx.x;
    const bool live = row_mask == nullptr || row_mask[row] != 0;
    const float p = live ? load_prob(probs, probs_bf16, row) : 0.f;
    const uint16_t* xg = x + row * 2 * f;
    const uint16_t* dyr = dy + row * f;
    uint16_t* dxr = dx + row * 2 * f;
    float sums[SUMS];
#pragma unroll
    for (int s = 0; s < SUMS; ++s) sums[s] = 0.f;
    int turn = 0;
    for (int64_t c = (int64_t)threadIdx.x * 8; c < f; c += THREADS * 8) {
        uint4 o1 = make_uint4(0, 0, 0, 0), o2 = o1;
        if (live) {
            const uint4 g = act_load16(xg + c), u = act_load16(xg + f + c), d = act_load16(dyr + c);
            const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w}, dw[4] = {d.x, d.y, d.z, d.w};
            uint32_t w1[4], w2[4];
            float acc = sums[0];
#pragma unroll
            for (int s = 1; s < SUMS; ++s) acc = turn == s ? sums[s] : acc;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float a0, da0, a1, da1;
                act_both<ACT>(bf16_lo(gw[k]), a0, da0);
                act_both<ACT>(bf16_hi(gw[k]), a1, da1);
                const float u0 = bf16_lo(uw[k]), u1 = bf16_hi(uw[k]);
                const float d0 = bf16_lo(dw[k]), d1 = bf16_hi(dw[k]);
                acc += d0 * (a0 * u0) + d1 * (a1 * u1);
                w1[k] = pack_bf16(d0 * p * u0 * da0, d1 * p * u1 * da1);
                w2[k] = pack_bf16(d0 * p * a0, d1 * p * a1);
            }
#pragma unroll
            for (int s = 0; s < SUMS; ++s) sums[s] = SUMS == 1 || turn == s ? acc : sums[s];
            turn = (turn + 1) & (SUMS - 1);
            o1 = make_uint4(w1[0], w1[1], w1[2], w1[3]);
            o2 = make_uint4(w2[0], w2[1], w2[2], w2[3]);
        }
        act_store16(dxr + c, o1);
        act_store16(dxr + f + c, o2);
    }
    // row sum of dy * act(g) * u over the workgroup
#pragma unroll
    for (int i = 0; i < SUMS; ++i) {
        float acc = sums[i];
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
        if ((threadIdx.x & 63) == 0) part[i * (THREADS / 64) + (threadIdx.x >> 6)] = acc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < SUMS * THREADS / 64; ++i) t += part[i];
        dprobs[row] = live ? t : 0.f;
    }
}

}  // namespace mxl

using namespace mxl;

static bool act_args_ok(const void* a, const void* b, const void* probs, int probs_dtype, int64_t rows, int64_t f, int act) {
    if (rows < 0 || f <= 0 || f % 8 != 0 || rows > 0x7FFFFFFF) return false;
    if (act != MXL_ACT_SILU && act != MXL_ACT_GELU) return false;
    if (probs_dtype != MXL_PROBS_F32 && probs_dtype != MXL_PROBS_BF16) return false;
    return rows == 0 || (a && b && probs);
}

// mask[i] = i < sum of the lens: which rows of a buffer sized for the worst case hold tokens.  A few kilobytes, so the launch is
// all it costs: one instead of the three of a sum, a range and a comparison (32 groups, 8192 rows: 15.4 -> 6.7 us).
constexpr int MASK_ROWS = 16;      // rows per thread, one 16-byte store
__global__ __launch_bounds__(ATHREADS) void row_mask_kernel(const int64_t* lens, int64_t count, int64_t rows, uint8_t* mask) {
    __shared__ int64_t part[ATHREADS / 64];
    const int t = threadIdx.x;
    int64_t sum = 0;
    for (int64_t i = t; i < count; i += ATHREADS) sum += lens[i];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s);
    if ((t & 63) == 0) part[t >> 6] = sum;
    __syncthreads();
    sum = 0;
#pragma unroll
    for (int w = 0; w < ATHREADS / 64; ++w) sum += part[w];
    const int64_t row0 = ((int64_t)blockIdx.x * ATHREADS + t) * MASK_ROWS;
    if (row0 + MASK_ROWS <= rows) {
        uint32_t v[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < MASK_ROWS; ++j) v[j >> 2] |= (row0 + j < sum ? 1u : 0u) << (8 * (j & 3));
        *(uint4*)(mask + row0) = make_uint4(v[0], v[1], v[2], v[3]);
    } else {
        for (int64_t i = row0; i < rows; ++i) mask[i] = i < sum ? 1 : 0;
    }
}

extern "C" int mxl_row_mask(const int64_t* lens, int64_t count, int64_t rows, uint8_t* mask, void* stream) {
    if (count < 1 || rows < 0 || !lens || (rows > 0 && !mask) || ((uintptr_t)mask & 15) != 0) return MXL_EINVAL;
    if (rows == 0) return MXL_OK;
    const int64_t grid = (rows + ATHREADS * MASK_ROWS - 1) / (ATHREADS * MASK_ROWS);
    if (grid > 0x7FFFFFFF) return MXL_EINVAL;
    if (!device_is_gfx950()) return MXL_ENODEV;
    hipLaunchKernelGGL(row_mask_kernel, dim3((unsigned)grid), dim3(ATHREADS), 0, (hipStream_t)stream, lens, count, rows, mask);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

template <int ACT, int THREADS>
static void launch_glu_fwd(const void* x, const void* probs, int probs_dtype, const uint8_t* row_mask, int64_t rows, int64_t f, void* y, hipStream_t st) {
    hipLaunchKernelGGL((glu_probs_fwd_kernel<ACT, THREADS>), dim3((unsigned)rows), dim3(THREADS), 0, st, (const uint16_t*)x, probs, probs_dtype, row_mask,
                       f, (uint16_t*)y);
}
template <int ACT, int THREADS, int SUMS>
static void launch_glu_bwd(const void* dy, const void* x, const void* probs, int probs_dtype, const uint8_t* row_mask, int64_t rows, int64_t f,
                           void* dx, void* dprobs, hipStream_t st) {
    hipLaunchKernelGGL((glu_probs_bwd_kernel<ACT, THREADS, SUMS>), dim3((unsigned)rows), dim3(THREADS), 0, st, (const uint16_t*)dy, (const uint16_t*)x, probs,
                       probs_dtype, row_mask, f, (uint16_t*)dx, (float*)dprobs);
}
// 1024 threads from here on.  GELU, which computes more, has more than two passes of 512 threads in front of it: cold, 256 / 512 / 1024, forward
// [1890, 6656] 16.8 / 15.1 / 16.1, [7561, 6656] 53.8 / 49.5 / 51.4, [16384, 8192] 142 / 132 / 131; backward 31.9 / 30.4 / 30.8, 107 / 104 / 108,
// 273 / 276 / 281, and beyond [9830, 10240] 210 / 208 / 211, [585, 14336] 27.2 / 23.7 / 22.7.
constexpr int64_t GLU_LONG_ROW[2] = {6656, 8200};
// 512 threads.  The forward of 4096 columns is whole passes of 256 threads: cold, 256 / 512, [2197, 4096] 13.0 / 14.1, [1098, 4096] 9.0 / 9.6,
// [14160, 4096] 58.6 / 57.8, and one chunk more [2192, 4104] 14.0 / 14.0, [14132, 4104] 62.4 / 58.4.
constexpr int64_t GLU_FWD_MIDDLE_ROW = 4104, GLU_BWD_MIDDLE_ROW = 2560;
// A workgroup takes half the threads its row's length gives it where whole workgroups are more waves than the chip holds (32 to a CU: 8192) and
// halves are not, on rows that fill the halves' passes.  SILU, us, half / whole: backward [1638, 2560] 10.2 / 10.6, [1170, 3584] 10.2 / 10.8, [1536, 4096] 13.4 /
// 14.0, [2048, 4096] 16.6 / 16.9, [768, 8192] 13.5 / 14.4, [1024, 8192] 17.4 / 17.9, but [1092, 2880] 9.2 / 8.9, [2184, 2880] 14.5 / 14.0, [1456, 5760]
// 18.0 / 17.4; forward [768, 8192] 8.5 / 8.9, [1024, 8192] 10.6 / 11.0.  GELU loses: backward [1638, 2560] 12.8 / 12.2, [768, 8192] 16.2 / 15.7.
static bool glu_halves(int act, int64_t rows, int64_t f) {
    if (act != MXL_ACT_SILU) return false;
    return f >= GLU_LONG_ROW[act] ? f <= 8192 && rows > 512 && rows <= 1024 : f <= 4096 && rows > 1152 && rows <= 2048;
}

extern "C" int mxl_glu_probs_fwd(const void* x_bf16, const void* probs, int probs_dtype, const uint8_t* row_mask,
                                 int64_t rows, int64_t f, int act, void* y_bf16, void* stream) {
    if (!act_args_ok(x_bf16, y_bf16, probs, probs_dtype, rows, f, act)) return MXL_EINVAL;
    if (rows == 0) return MXL_OK;
    if (!device_is_gfx950()) return MXL_ENODEV;
    const bool silu = act == MXL_ACT_SILU;
    const auto launch = f >= GLU_LONG_ROW[act] && !glu_halves(act, rows, f) ? (silu ? launch_glu_fwd<MXL_ACT_SILU, 1024> : launch_glu_fwd<MXL_ACT_GELU, 1024>)
                        : f >= GLU_FWD_MIDDLE_ROW ? (silu ? launch_glu_fwd<MXL_ACT_SILU, 512> : launch_glu_fwd<MXL_ACT_GELU, 512>)
                                                  : (silu ? launch_glu_fwd<MXL_ACT_SILU, 256> : launch_glu_fwd<MXL_ACT_GELU, 256>);
    launch(x_bf16, probs, probs_dtype, row_mask, rows, f, y_bf16, (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}

namespace mxl {
// `shared`: another launch that fills the chip runs on another stream.  Its workgroups leave room here and there, which small
// workgroups use better: a pass of 8 experts [28672, 4096] and [4096, 14336] whose weight gradients run beside it, with 256 threads
// (and four sums each) and with 1024: FP8, 32768 rows, 16.00 and 16.23 ms; E2M1, 8192 rows, 3.69 and 3.73.
int glu_probs_bwd(const void* dy_bf16, const void* x_bf16, const void* probs, int probs_dtype, const uint8_t* row_mask, int64_t rows, int64_t f, int act,
                  void* dx_bf16, void* dprobs_f32, bool shared, void* stream) {
    if (!act_args_ok(x_bf16, dx_bf16, probs, probs_dtype, rows, f, act)) return MXL_EINVAL;
    if (rows == 0) return MXL_OK;
    if (!dy_bf16 || !dprobs_f32) return MXL_EINVAL;
    if (!device_is_gfx950()) return MXL_ENODEV;
    const bool silu = act == MXL_ACT_SILU;
    const bool halves = glu_halves(act, rows, f);
    const auto launch =
        f >= GLU_LONG_ROW[act]  ? (shared ? (silu ? launch_glu_bwd<MXL_ACT_SILU, 256, 4> : launch_glu_bwd<MXL_ACT_GELU, 256, 4>)
                                 : halves ? launch_glu_bwd<MXL_ACT_SILU, 512, 2>
                                          : (silu ? launch_glu_bwd<MXL_ACT_SILU, 1024, 1> : launch_glu_bwd<MXL_ACT_GELU, 1024, 1>))
        : f >= GLU_BWD_MIDDLE_ROW ? (shared || halves ? (silu ? launch_glu_bwd<MXL_ACT_SILU, 256, 2> : launch_glu_bwd<MXL_ACT_GELU, 256, 2>)
                                          : (silu ? launch_glu_bwd<MXL_ACT_SILU, 512, 1> : launch_glu_bwd<MXL_ACT_GELU, 512, 1>))
                                : (silu ? launch_glu_bwd<MXL_ACT_SILU, 256, 1> : launch_glu_bwd<MXL_ACT_GELU, 256, 1>);
    launch(dy_bf16, x_bf16, probs, probs_dtype, row_mask, rows, f, dx_bf16, dprobs_f32, (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? MXL_OK : MXL_ELAUNCH;
}
}  // namespace mxl

extern "C" int mxl_glu_probs_bwd(const void* dy_bf16, const void* x_bf16, const void* probs, int probs_dtype,
                                 const uint8_t* row_mask, int64_t rows, int64_t f, int act, void* dx_bf16,
                                 void* dprobs_f32, void* stream) {
    return mxl::glu_probs_bwd(dy_bf16, x_bf16, probs, probs_dtype, row_mask, rows, f, act, dx_bf16, dprobs_f32, false, stream);
}
