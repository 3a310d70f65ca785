// Quants to exact f16 or bf16 MFMA fragments, shared by the prefill GEMMs.
#pragma once

#include "common.h"

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ uint32_t as_u32(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// XOR swizzles of the 16-byte chunks of an LDS tile's rows, so that the rows of a
// fragment read fall in distinct bank groups: f16 activations or weights (128 B
// rows of 64 values), Q8_0 quants (64 B) and Q4_0 quants (32 B).
__device__ __forceinline__ int swz_a(int r) { return (r & 7) ^ ((r >> 1) & 4); }
__device__ __forceinline__ int swz_q8(int r) { return (r >> 2) & 3; }
__device__ __forceinline__ int swz_q4(int r) { return (r >> 3) & 1; }

// 4 signed bytes -> 2 dwords holding the 4 quants as f16 pairs (exact).
__device__ __forceinline__ void int8x4_to_f16(uint32_t w, uint32_t& o0, uint32_t& o1) {
    const uint32_t u = w ^ 0x80808080u;  // q + 128 in each byte
    const h2 bias = {(f16)1152.0f, (f16)1152.0f};
    o0 = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - bias);
    o1 = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - bias);
}
// 4 nibbles (one per byte, already masked) -> nib - 8 as f16 pairs (exact).
__device__ __forceinline__ void nib4_to_f16(uint32_t nib, uint32_t& o0, uint32_t& o1) {
    const h2 bias = {(f16)1032.0f, (f16)1032.0f};
    o0 = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, nib, 0x04010400u)) - bias);
    o1 = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, nib, 0x04030402u)) - bias);
}
// The same as bf16 pairs: the top halves of their float32 values (exact).
__device__ __forceinline__ void int8x4_to_bf16(uint32_t w, uint32_t& o0, uint32_t& o1) {
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; e++) f[e] = (float)(int8_t)(w >> (8 * e));
    o0 = __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u);
    o1 = __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u);
}
__device__ __forceinline__ void nib4_to_bf16(uint32_t nib, uint32_t& o0, uint32_t& o1) {
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; e++) f[e] = (float)((nib >> (8 * e)) & 255u) - 8.0f;
    o0 = __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u);
    o1 = __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u);
}
