// What the attention kernels of MLA.forward share: bf16 MFMAs of 32 x 32, copies into LDS, masks, the softmax offset.
#pragma once
#include <type_traits>
#include "common.hpp"

namespace dsv3 {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lptr_t;

__device__ __forceinline__ v16f mfma32(v4u a, v4u b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t lds_addr_of(const void* p) { return (uint32_t)(uintptr_t)(lptr_t)p; }
// 1 KiB global -> LDS: lane l's 16 bytes at base + lane_off land at lds_addr + 16 l
__device__ __forceinline__ void copy16(const void* base, uint32_t lane_off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(lane_off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
// The same through a buffer descriptor (the range check answers requests past its end with zeros), into LDS at lds_addr + IMM
__device__ __forceinline__ v4i buffer_of(const void* base, int bytes) {
    const uintptr_t a = (uintptr_t)base;
    return v4i{ (int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xffffu), bytes, 0x00027000 };
}
template <int IMM> __device__ __forceinline__ void copy16_buffer(v4i buffer, uint32_t lane_off, uint32_t lds_addr) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 :: "v"(lane_off), "s"(buffer), "s"(lds_addr), "n"(IMM) : "memory", "m0", "scc");
}
// f(integral_constant 0), .., f(integral_constant N - 1)
template <int N, int I = 0, class F> __device__ __forceinline__ void unrolled(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        unrolled<N, I + 1>(f);
    }
}
__device__ __forceinline__ void barrier_no_fence() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ float xor32(float v) { return __shfl_xor(v, 32); }
// the values of lanes l and l + 32, in this order, in both
__device__ __forceinline__ v2f halves32(float v) {
    const v2u r = __builtin_amdgcn_permlane32_swap(f32_as_u32(v), f32_as_u32(v), false, false);
    return v2f{ u32_as_f32(r[0]), u32_as_f32(r[1]) };
}

template <bool F32> __device__ __forceinline__ float mask_at(const void* m, int64_t i) {
    return F32 ? ((const float*)m)[i] : u32_as_f32((uint32_t)((const uint16_t*)m)[i] << 16);
}
// The unit in which scores are kept beside a mask: the raw ones times the largest power of two that is not above the
// softmax scale (1 for scales above 1), scale = unit * rest.  The power of two costs no rounding, and a mask value, which
// counts in units of scale, is divided by a rest of at least 1: every finite one stays finite and keeps its order.  (That
// quotient is rounded before the score is added: equal mask values of a size that swallows the scores must stay equal.)
struct ScoreUnit { float unit, rest; };
inline ScoreUnit score_unit(float scale) {
    int e;
    const float m = __builtin_frexpf(scale, &e);        // m * 2^e, m in [1/2, 1)
    return scale < 1.f ? ScoreUnit{ __builtin_ldexpf(1.f, e - 1), 2.f * m } : ScoreUnit{ 1.f, scale };
}
// What the exponents fma(S, scale2, -offset) subtract for a row maximum m.  Where the maximum is huge (a row that only
// finite mask values of such a size reach), the rounding of m * scale2 alone would overflow the exponentials: the maximum
// is taken off the scores themselves then.
template <int N> __device__ __forceinline__ float softmax_offset(v16f (&S)[N], float m, float scale2) {
    float off = m == -__builtin_inff() ? 0.f : m * scale2;
    const bool huge = __builtin_fabsf(m) > 0x1p20f && m != -__builtin_inff();
    if (__any(huge)) {
        const float d = huge ? m : 0.f;
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int e = 0; e < 16; ++e) S[k][e] -= d;
        off = huge ? 0.f : off;
    }
    return off;
}

}  // namespace
}  // namespace dsv3
