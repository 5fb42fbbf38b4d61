// What the MX GEMM kernels share: the launch arguments and the LDS-direct loads.
#pragma once
#include <type_traits>

#include "mx_device.h"
#include "mx_gemm_addr.h"

namespace mxl {

constexpr int BM = 256, BN = 256;
constexpr int BK = 64;     // one MFMA K step (two MX blocks)
constexpr int GTHREADS = 256;
constexpr int MODE_FWD = 0;    // rows of A ragged by group; B = [G, N, K]
constexpr int MODE_WGRAD = 1;  // contraction ragged by group; C = [G, M, N]
constexpr int GROUP_M = 4;     // tile-order super-row height (L2 locality)

struct GemmArgs {
    const uint8_t* a;   // M-side codes
    const uint8_t* sa;  // M-side scales
    const uint8_t* b;   // N-side codes
    const uint8_t* sb;  // N-side scales
    uint16_t* c;        // bf16 out
    const int64_t* group_lens;  // device, may be null (one group)
    int num_groups;     // >= 1
    int64_t total_m;    // FWD: rows of a; WGRAD: tokens (sum of lens)
    int64_t m;          // WGRAD: rows of a (fixed)   | FWD: unused
    int64_t n;          // columns of c / rows of b
    int64_t b_rows;     // FWD: rows from one group's matrix in b to the next (n, or more where the matrices are padded)
    int64_t k;          // FWD: contraction length; WGRAD: padded width W
    const float* alpha_a;   // ALPHA kernels: the output is multiplied by *alpha_a * *alpha_b (per-tensor
    const float* alpha_b;   // scales of tensor-wise quantised operands) before it is rounded
};

// ---- asynchronous global -> LDS loads ------------------------------------
// Written as inline assembly on purpose: the compiler then keeps no record of
// LDS writes in flight and does not put a full vmcnt wait in front of every
// LDS read; completion is waited for explicitly (wait_vm) before the barrier
// that publishes a stage.  The hardware writes lane i's data to LDS address
// M0 + size*i, so the XOR swizzle is applied on the global side: the lane that
// owns physical chunk (row, pch) fetches logical chunk pch ^ swz(row).
__device__ __forceinline__ v4i make_rsrc(const void* base, int64_t bytes) {
    const uint64_t p = (uint64_t)base;
    const uint32_t n = bytes > 0xFFFFFFFFll ? 0xFFFFFFFFu : (uint32_t)(bytes < 0 ? 0 : bytes);
    v4i r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32) & 0xFFFF);  // stride 0: raw buffer
    r[2] = __builtin_amdgcn_readfirstlane((int)n);                             // bytes; reads past it give 0
    r[3] = 0x00020000;
    return r;
}
// The statement writes M0 (the LDS address of an LDS-direct load).  M0 cannot be named in the clobber list: the
// compiler diagnoses clobbers of reserved registers.  Nothing else in these kernels lives in M0: LDS instructions do
// not take it on gfx950 and the kernels use no relative moves, messages or interpolation, and every use here
// reloads it first.
__device__ __forceinline__ void dma16(v4i rsrc, uint32_t lds_off, uint32_t voff, uint32_t soff) {
    asm volatile("" : "+s"(soff));   // the scalar offset has to sit in a register, also when it is a known constant
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_off), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// The same load with the LDS address formed in M0 by one scalar add (base register + constant) and the scalar
// offset taken as it is: the ring kernel keeps a round's row offset in the per-lane offset instead of adding it to
// the scalar one, which leaves two scalar instructions per request.
template <int LDS_IMM>
__device__ __forceinline__ void dma16_at(v4i rsrc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                 :
                 : "s"(lds_base), "n"(LDS_IMM), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "scc");
}

// Output stores are marked non-temporal: the kernel never reads its output back, and keeping it
// out of the way leaves L2 to the operand tiles that neighbouring workgroups share.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store16_streaming(uint8_t* dst, const uint4& v) {
    const u32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, (u32x4*)dst);
}

// The same through a buffer descriptor (base and size uniform): a lane whose offsets pass its end stores nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_store_rsrc(void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
}
// A store of more than 8 bytes fetches its data registers after it has issued: an instruction right behind it that writes
// one of them changes what is stored, in some lanes and now and then (seen as single wrong dwords in lanes 12-15, 28-31, ..
// of a store directly followed by a multiplication into its first data register).  The compiler puts the wait states in for
// a store without a scalar offset register only, so they are written here: the statement takes the data as an operand, so
// the registers cannot be handed on before it.
__device__ __forceinline__ void buffer_store16_streaming(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, const uint4& v) {
    const u32x4 t = {v.x, v.y, v.z, v.w};
    constexpr int kNonTemporal = 2;
    __builtin_amdgcn_raw_buffer_store_b128(t, rsrc, (int)voff, (int)soff, kNonTemporal);
    asm volatile("s_nop 1" : : "v"(t) : "memory");
}

// compile-time loop: f(integral_constant<int, I>) for I .. N - 1
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

}  // namespace mxl
