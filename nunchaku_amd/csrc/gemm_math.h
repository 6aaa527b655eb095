// Device code that the GEMM kernels share: the matrix instructions on INT4 codes, the NVFP4 dequantization, the GELU.
#pragma once

#include "svdq_common.h"

namespace svdq {

// ---- INT4: E2M3 code fragments (svdq_common.h) ----------------------------------------------------
typedef int v8i_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

struct Frag {
    u32x4_t lo;  // bits [0, 128) of the lane's 192-bit code string
    u32x2_t hi;  // bits [128, 192)
};

typedef int v6i_t __attribute__((ext_vector_type(6)));
__device__ inline v6i_t codes6(u32x4_t lo, u32x2_t hi) { return v6i_t{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1]}; }

// inner sums of one 32 x 32 tile over one k-group (elements 6 and 7 of the operand vectors are not
// read by the fp6 form of the instruction)
__device__ inline float16_t mfma_codes6(v6i_t w, v6i_t x) {
    const v8i_t a = __builtin_shufflevector(w, w, 0, 1, 2, 3, 4, 5, -1, -1), b = __builtin_shufflevector(x, x, 0, 1, 2, 3, 4, 5, -1, -1);
    const float16_t z = {};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, z, 2, 2, 0, 0, 0, 0);  // E2M3 x E2M3, no block scales
}
__device__ inline float16_t mfma_codes(const Frag &w, const Frag &x) { return mfma_codes6(codes6(w.lo, w.hi), codes6(x.lo, x.hi)); }

// factor tile 64 ws[n] * as[m]: the weight operand is {64 s, 0, 0, 0} in both half-waves (k slots 0-3 and
// 4-7), the activation operand carries its scale in k slot 0 and zero in k slot 4, anything finite
// elsewhere.  (A pair of registers whose second one stays zero: put together from a scale and a zero, the operand costs the
// caller up to two instructions each time.)
__device__ inline float16_t mfma_factor(u32x2_t ws, u32x2_t as) {
    const float16_t z = {};
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(bf16x4_t, ws), __builtin_bit_cast(bf16x4_t, as), z, 0, 0, 0);
}

// ---- NVFP4 ------------------------------------------------------------------------------------------
__device__ inline half2_t as_half2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }
__device__ inline uint32_t as_u32(half2_t h) { return __builtin_bit_cast(uint32_t, h); }

// 8 E2M1 patterns of one word -> 8 fp16 values pattern_value * scale, slot order [0..7].  The
// hardware conversion yields the exact E2M1 value (its scale operand only contributes an exponent).
template <int PAIR>
__device__ inline half2_t dequant_pair_fp4(uint32_t w, half2_t s) {
    return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, PAIR) * s;
}
__device__ inline half8_t dequant_word_fp4(uint32_t w, half2_t s) {
    const half2_t t0 = dequant_pair_fp4<0>(w, s), t1 = dequant_pair_fp4<1>(w, s), t2 = dequant_pair_fp4<2>(w, s), t3 = dequant_pair_fp4<3>(w, s);
    return half8_t{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
}

__device__ inline float gelu_tanh(float x) {
    // x * (0.5 + 0.5 * tanh(u)), u = 0.79788456 * (x + 0.044715 x^3)   (epilogues.cuh:22-44)
    // With tanh(u) = 1 - 2 / (exp(2u) + 1) this is x - x / (exp(2u) + 1): one hardware exp2 and one hardware
    // reciprocal (1 ulp each), safe at both ends (exp2 -> inf gives x, exp2 -> 0 gives 0).
    constexpr float C1 = 2.0f * 0.79788456f * 1.4426950408889634f, C2 = C1 * 0.044715f;  // 2u * log2(e) = x (C1 + C2 x^2)
    const float w = x * __builtin_fmaf(C2, x * x, C1);
    const float r = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(w) + 1.0f);
    return __builtin_fmaf(-x, r, x);
}

}  // namespace svdq
