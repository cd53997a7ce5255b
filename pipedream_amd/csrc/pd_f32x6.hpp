// Pieces shared by the kernels that keep a whole operand fragment in registers and multiply fp32 values on the bf16
// matrix pipes: x = x1 + x2 + x3 exactly (three bf16 terms), a b = a3 b1 + a1 b3 + a2 b2 + a2 b1 + a1 b2 + a1 b1 up to
// 2^-24 a b (pd_gemm_f32x6.hip has the derivation; there the terms pass through LDS).
#pragma once
#include "pd_internal.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// (the instruction itself: from two conversions the compiler makes an instruction per use of a half)
__device__ __forceinline__ uint32_t pd_x6_pack(float lo, float hi) {
    uint32_t p;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(p) : "v"(lo), "v"(hi));
    return p;
}

// the three terms of two neighbouring values, as one packed dword each
__device__ __forceinline__ void pd_x6_split2(float x0, float x1, uint32_t& t1, uint32_t& t2, uint32_t& t3) {
    t1 = pd_x6_pack(x0, x1);
    const float r0 = x0 - __builtin_bit_cast(float, t1 << 16), r1 = x1 - __builtin_bit_cast(float, t1 & 0xffff0000u);
    t2 = pd_x6_pack(r0, r1);
    t3 = pd_x6_pack(r0 - __builtin_bit_cast(float, t2 << 16), r1 - __builtin_bit_cast(float, t2 & 0xffff0000u));
}

// the three terms of the eight consecutive k of one lane
__device__ __forceinline__ void pd_x6_split8(const float (&x)[8], u32x4_t (&t)[3]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t a, b, c;
        pd_x6_split2(x[2 * q], x[2 * q + 1], a, b, c);
        t[0][q] = a;
        t[1][q] = b;
        t[2][q] = c;
    }
}

// which term of A meets which term of B, small products first
constexpr int PD_X6_A[6] = {2, 0, 1, 1, 0, 0};
constexpr int PD_X6_B[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ f32x4_t pd_x6_mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
