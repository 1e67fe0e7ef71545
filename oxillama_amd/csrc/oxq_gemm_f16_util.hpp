// Pieces shared by the matmul kernels that run on the f16 matrix cores (oxq_gemm_prefill.hip, oxq_gemm_f16.hip).
#pragma once
#include <utility>
#include "oxq_gemm_tile.hpp"

namespace oxq {

template <class F, int... Q>
__device__ __forceinline__ void static_for(std::integer_sequence<int, Q...>, F &&f) {
    (f(std::integral_constant<int, Q>{}), ...);
}

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

#define OXQ_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

// LDS is carved out of byte arrays here and written with one vector type and read with another (and filled by
// direct-to-LDS loads): every such access goes through a may_alias type, or type-based alias analysis treats a
// load as unrelated to the store that feeds it.
typedef u32x4 __attribute__((may_alias)) lds_u32x4;
typedef u32x2 __attribute__((may_alias)) lds_u32x2;
typedef uint32_t __attribute__((may_alias)) lds_u32;
typedef uint16_t __attribute__((may_alias)) lds_u16;
typedef float __attribute__((may_alias)) lds_f32;
typedef v4f __attribute__((may_alias)) lds_v4f;
__device__ __forceinline__ h8 lds_h8(const uint8_t *p) { return __builtin_bit_cast(h8, *reinterpret_cast<const lds_u32x4 *>(p)); }
__device__ __forceinline__ b8 lds_b8(const uint8_t *p) { return __builtin_bit_cast(b8, *reinterpret_cast<const lds_u32x4 *>(p)); }

// Order of the eight k-slots of one operand register set: byte positions of the lane's 8 raw weight bytes.  The
// unpack takes bytes 0 and 2 of a dword together (they sit in the two 16-bit halves), then bytes 1 and 3.
__device__ __forceinline__ constexpr int pf_slot_byte(int j) { return (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1); }

// The bits of three truncated bf16 pieces whose sum is x, exact for up to 23 significant bits.  A piece that is x itself
// leaves no rest: of an infinity, x - x would be a NaN.
__device__ __forceinline__ void bf16_pieces(float x, uint16_t (&piece)[3]) {
    const uint32_t p1 = __builtin_bit_cast(uint32_t, x) & 0xFFFF0000u;
    const float f1 = __builtin_bit_cast(float, p1);
    const float r1 = x == f1 ? 0.0f : x - f1;  // exact
    const uint32_t p2 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
    const float r2 = r1 - __builtin_bit_cast(float, p2);  // exact, at most 8 significant bits
    piece[0] = (uint16_t)(p1 >> 16);
    piece[1] = (uint16_t)(p2 >> 16);
    piece[2] = (uint16_t)(__builtin_bit_cast(uint32_t, r2) >> 16);
}

__device__ __forceinline__ uint32_t f16x2_of(float v) {
    const uint32_t b = f2h(v);
    return b | (b << 16);
}

}  // namespace oxq
