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
// Splitting.  The difference x - h of an infinite h counts as 0.
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

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// x - h for the halves of a packed pair, exact.  fp16: one mixed FMA each.
__device__ __forceinline__ void sub_pair(FmtF16, unsigned h, float x0, float x1, float &r0, float &r1) {
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(h), "v"(x0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(h), "v"(x1));
}
__device__ __forceinline__ void sub_pair(FmtBf16, unsigned h, float x0, float x1, float &r0, float &r1) {
    r0 = x0 - __uint_as_float(h << 16);
    r1 = x1 - __uint_as_float(h & 0xffff0000u);
}

// Some of the 8 values of a row may become infinite in the 16-bit format:
// the quick split below doesn't hold.  bf16: by the largest magnitude, from
// half a step above the largest bf16 (a NaN among them is passed over: its
// row's results are NaN whatever the others split into).  fp16: where the
// row's largest magnitude is infinite (finite ones scale below 2^15).
__device__ __forceinline__ bool split_special(FmtBf16, const float (&x)[8], bool) {
    float m;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(m) : "v"(x[0]), "v"(x[1]), "v"(x[2]));
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(m) : "v"(m), "v"(x[3]), "v"(x[4]));
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(m) : "v"(m), "v"(x[5]), "v"(x[6]));
    asm("v_max3_f32 %0, %1, |%2|, |%2|" : "=v"(m) : "v"(m), "v"(x[7]));
    return !(m < __uint_as_float(0x7f7f8000u));
}
__device__ __forceinline__ bool split_special(FmtF16, const float (&)[8], bool row_inf) { return row_inf; }
__device__ __forceinline__ bool row_is_inf(unsigned amax_bits) { return amax_bits == 0x7f800000u; }

// The NP planes of 8 values of one row.  special: some lane's values are (any
// lane's answer of split_special, wave-uniform).  The quick form takes 24
// instructions (bf16, two planes) or 16 (fp16), the general one 49 and 40,
// which the cores that split an operand and the small grids wait for: 512
// grouped FP16X3 problems 3.68 ms of core before, 3.17 after (with the loads
// at edges, load_rc); 1024x1024x1024 FP16X3 NN 33 us and 30.
template <int NP, class FMT>
__device__ __forceinline__ void split8(const float (&x)[8], bool special, typename FMT::V8 (&w)[NP]) {
    using V8 = typename FMT::V8;
    typedef float f8 __attribute__((ext_vector_type(8)));
    if (NP > 1 && special) {
        typename FMT::E o[NP][8];
        split_vec<NP, 8>(x, o);
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int j = 0; j < 8; ++j) w[p][j] = o[p][j];
        return;
    }
    f8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = x[j];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        w[p] = __builtin_convertvector(v, V8);
        if (p + 1 < NP) {
            const u32x4 h = __builtin_bit_cast(u32x4, w[p]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float r0, r1;
                sub_pair(FMT(), h[j], v[2 * j], v[2 * j + 1], r0, r1);
                v[2 * j] = r0;
                v[2 * j + 1] = r1;
            }
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
