// MFMA input types of the BF16 / FP16 / split-BF16 kernels (device code,
// included by the .hip sources only).
#pragma once

#include "internal.h"

namespace cogconv {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

template <int PREC>
struct LpType;
template <>
struct LpType<COGCONV_BF16> {
    typedef __bf16 T;
    typedef bf16x8 V;
};
template <>
struct LpType<COGCONV_FP32> {  // as three BF16 terms
    typedef __bf16 T;
    typedef bf16x8 V;
};
template <>
struct LpType<COGCONV_SPLIT_BF16> {
    typedef __bf16 T;
    typedef bf16x8 V;
};
template <>
struct LpType<COGCONV_FP16> {
    typedef _Float16 T;
    typedef halfx8 V;
};

template <int PREC>
__device__ __forceinline__ floatx4 lp_mfma(typename LpType<PREC>::V a, typename LpType<PREC>::V b, floatx4 c) {
    if constexpr (PREC == COGCONV_FP16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Operands below this may lose bits of their last BF16 term (under 2^-126).
constexpr float LP_SMALL = 0x1p-102f;

// BF16 terms of an operand.
constexpr int lp_terms(int prec) { return prec == COGCONV_FP32 ? 3 : (prec == COGCONV_SPLIT_BF16 ? 2 : 1); }

// Splits x into T terms: term t rounds what the earlier ones left.
template <int T, class E>
__device__ __forceinline__ void split_terms(float x, E (&t)[T]) {
#pragma unroll
    for (int k = 0; k < T; k++) {
        t[k] = (E)x;
        if (k + 1 < T) x -= (float)t[k];
    }
}

__device__ __forceinline__ unsigned wave_max(unsigned v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, d));
    return v;
}

__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Whether any lane's operands go under LP_SMALL; `least`: the smallest magnitude(x) - 1, which puts zeros last.
__device__ __forceinline__ bool any_small(unsigned least) { return __any(least < __float_as_uint(LP_SMALL) - 1u); }

}  // namespace cogconv
