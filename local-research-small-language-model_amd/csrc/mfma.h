// gfx950 matrix-core helpers shared by the prefill and decode kernels:
// bf16 operand vectors, LDS operand reads (plain and transposed) and the
// lane-pair reductions over the row-swap permutes.
#pragma once

#include "common.h"

namespace sparda {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 lds_read8(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

// Transposed read (ds_read_b64_tr_b16). Within each 16-lane group, output
// lane i, element e is element i%4 of the 8-byte chunk addressed by lane
// 4e + i/4 of the group.
// The pointer is converted with an address-space cast (not through an integer)
// so that constant offsets from a common base fold into the instruction.
__device__ __forceinline__ i16x4 lds_read_tr(const uint16_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(const_cast<uint16_t*>(p)));
}

// max of m and 4 N accumulator values straight from the matrix cores, as
// compiler-visible instructions (v_maximum3_f32), so that the wait states a
// matrix result needs before a VALU reads it are placed by the compiler (for
// inline assembly it places none). A NaN among them gives NaN.
template <int N>
__device__ __forceinline__ float max_acc(const f32x4 (&s)[N], float m) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, s[n][0]), s[n][1]);
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, s[n][2]), s[n][3]);
    }
    return m;
}
// Reductions over lane pairs (l, l^16) and (l, l^32) with the gfx950 VALU
// row swaps: permlane16_swap(x, x) hands every lane the values of rows
// {2r, 2r+1} at its column, permlane32_swap(x, x) those of rows {r, r+2};
// both lanes of a pair combine the same two values in the same order.
// max with the lane 16 (SWAP16) or 32 lanes away. One asm block: a VALU write
// of a register needs two wait states before a permlane swap reads it, and the
// compiler does not count inline-assembly results as VALU writes, so the copy,
// the s_nop and the swap stay together.
__device__ __forceinline__ float pair16_max(float x) {
    float t;
    asm("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_max_f32 %0, %0, %1"
        : "+v"(x), "=&v"(t));
    return x;
}
__device__ __forceinline__ float pair32_max(float x) {
    float t;
    asm("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_max_f32 %0, %0, %1"
        : "+v"(x), "=&v"(t));
    return x;
}
__device__ __forceinline__ float pair16_sum(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pair32_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace sparda
