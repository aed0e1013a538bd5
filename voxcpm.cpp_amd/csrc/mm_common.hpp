// mm_common.hpp -- device helpers shared by the MUL_MAT kernels (mul_mat.hip, gemm_mid.hip): the matrix instruction, Q8_0
// bytes to f16 operands, direct loads into LDS, the residual update's rounding.
#pragma once
#include "vx_common.hpp"

namespace {

// a + x * s with the product rounded before the sum, as a SCALE node followed by an ADD node rounds
__device__ __forceinline__ float scaled_residual(float x, float s, float a) {
#pragma clang fp contract(off)
    const float t = x * s;
    return a + t;
}

__device__ __forceinline__ float4_t mfma16(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 8 int8 (two dwords) -> 8 f16, exactly
__device__ __forceinline__ half8_t q8_to_half8(uint32_t lo, uint32_t hi) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t bias = 0x64646464u;
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    u32x4 r;
    r[0] = __builtin_amdgcn_perm(bias, lo, 0x04010400u);
    r[1] = __builtin_amdgcn_perm(bias, lo, 0x04030402u);
    r[2] = __builtin_amdgcn_perm(bias, hi, 0x04010400u);
    r[3] = __builtin_amdgcn_perm(bias, hi, 0x04030402u);
    half8_t h = __builtin_bit_cast(half8_t, r);
    const _Float16 off = (_Float16) 1152.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] -= off;
    return h;
}

} // namespace
