// Element formats, splitting and products of the split forms (described in
// gemm_mfma.hip), shared by the plane-streaming core and the small-grid kernel.
#pragma once

#include "internal.h"
#include "kernel_common.h"

namespace ugemm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Element formats of the planes.
struct FmtBf16 {
    typedef __bf16 E;
    typedef bf16x8 V8;
    static constexpr bool SCALED = false;
    static constexpr const char *name = "bf16";
    __device__ static __forceinline__ floatx4 mfma(const V8 &a, const V8 &b, const floatx4 &c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
struct FmtF16 {
    typedef _Float16 E;
    typedef f16x8 V8;
    static constexpr bool SCALED = true;
    static constexpr const char *name = "fp16";
    __device__ static __forceinline__ floatx4 mfma(const V8 &a, const V8 &b, const floatx4 &c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// Scale exponent of a row from the bit pattern of its largest magnitude:
// x * 2^-row_exp lies in (-2^15, 2^15).  0, inf and NaN give -15 (the
// products are then 0 or non-finite whatever the scale).
__device__ __forceinline__ int row_exp(unsigned amax_bits) {
    int e = 0;
    const float a = __uint_as_float(amax_bits);
    if (a != 0.0f && __builtin_isfinite(a)) frexpf(a, &e);
    return e - 15;
}

// ---------------------------------------------------------------------------
// Splitting.
template <int NP, int W, class E>
__device__ __forceinline__ void split_vec(const float (&x)[W], E (&out)[NP][W]) {
    typedef float fv __attribute__((ext_vector_type(W)));
    typedef E bv __attribute__((ext_vector_type(W)));
    fv v;
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = x[i];
    bv h = __builtin_convertvector(v, bv);
#pragma unroll
    for (int i = 0; i < W; ++i) out[0][i] = h[i];
    if constexpr (NP > 1) {
        fv hf = __builtin_convertvector(h, fv);
        fv r;
#pragma unroll
        for (int i = 0; i < W; ++i) r[i] = __builtin_isfinite(hf[i]) ? v[i] - hf[i] : 0.0f;
        bv l = __builtin_convertvector(r, bv);
#pragma unroll
        for (int i = 0; i < W; ++i) out[1][i] = l[i];
        if constexpr (NP > 2) {
            fv lf = __builtin_convertvector(l, fv);
            fv r2 = r - lf;
            bv l2 = __builtin_convertvector(r2, bv);
#pragma unroll
            for (int i = 0; i < W; ++i) out[2][i] = l2[i];
        }
    }
}

template <int NP>
struct Products;
template <>
struct Products<1> {
    static constexpr int N = 1;
    static constexpr int a[1] = {0}, b[1] = {0};
};
template <>
struct Products<2> {
    static constexpr int N = 3;
    static constexpr int a[3] = {1, 0, 0}, b[3] = {0, 1, 0};
};
template <>
struct Products<3> {
    static constexpr int N = 6;
    static constexpr int a[6] = {2, 0, 1, 1, 0, 0}, b[6] = {0, 2, 1, 0, 1, 0};
};

}  // namespace
}  // namespace ugemm
