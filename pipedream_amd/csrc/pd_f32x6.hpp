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

// the three terms of two neighbouring values, as one packed dword each; SIGNED: of the values times sign (1 or -1)
template <bool SIGNED = false>
__device__ __forceinline__ void pd_x6_split2(float x0, float x1, uint32_t& t1, uint32_t& t2, uint32_t& t3, float sign = 1.f) {
    t1 = pd_x6_pack(x0, x1);
    if (SIGNED) t1 ^= sign < 0.f ? 0x80008000u : 0u;
    const float h0 = __builtin_bit_cast(float, t1 << 16), h1 = __builtin_bit_cast(float, t1 & 0xffff0000u);
    const float r0 = SIGNED ? __builtin_fmaf(x0, sign, -h0) : x0 - h0, r1 = SIGNED ? __builtin_fmaf(x1, sign, -h1) : x1 - h1;
    t2 = pd_x6_pack(r0, r1);
    t3 = pd_x6_pack(r0 - __builtin_bit_cast(float, t2 << 16), r1 - __builtin_bit_cast(float, t2 & 0xffff0000u));
}

// the three terms of the eight consecutive k of one lane
template <bool SIGNED = false>
__device__ __forceinline__ void pd_x6_split8(const float (&x)[8], u32x4_t (&t)[3], float sign = 1.f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t a, b, c;
        pd_x6_split2<SIGNED>(x[2 * q], x[2 * q + 1], a, b, c, sign);
        t[0][q] = a;
        t[1][q] = b;
        t[2][q] = c;
    }
}

// v_mfma_f32_16x16x32_bf16 rounds its sums towards minus infinity: half an ulp of the same sign in every addition, which
// adds up in what sums over the results.  So the waves that share a reduction take turns at summing up the product and
// its negative: the sign of way `way` of `ways` over `chunks` chunks (ways without a chunk do not count).  2-norm errors,
// fp32 MFMAs / one sign / two: LSTM bias gradients over 50 steps of 128 sentences 1.6e-7 / 4.0e-7 / 1.5e-7, row sums of
// 64 x 4096 x 25088 7.4e-7 / 1.2e-5 / 4.9e-7; it costs a vector instruction per pair of values (GNMT stage 0.6 %).
__device__ __forceinline__ float pd_x6_sign(int chunks, int ways, int way) {
    return (chunks >= ways ? way : chunks * way / ways) & 1 ? -1.f : 1.f;
}

// which term of A meets which term of B, small products first
constexpr int PD_X6_A[6] = {2, 0, 1, 1, 0, 0};
constexpr int PD_X6_B[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ f32x4_t pd_x6_mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
