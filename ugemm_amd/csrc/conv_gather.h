// Gather of an implicit im2col operand tile (ConvDesc) for the FP32 vector and
// FP32-MFMA tiles: BK rows k of BN columns n, NT threads, one column per
// thread and rows k = t / BN + i * (NT / BN), the same for all lanes of a wave.
#pragma once

#include "internal.h"

namespace ugemm {
namespace {

static __device__ const float kConvZero = 0.0f;   // what an element outside the image reads

template <int BK, int BN, int NT>
struct ConvRegs {
    static_assert(NT % BN == 0 && BN % 64 == 0, "one column per thread, one k per wave");
    static constexpr int NE = BK * BN / NT, KSTEP = NT / BN;
    float v[NE];
    int base, h0, w0;      // offset of tap (0, 0) in its channel, and where it lies
    unsigned taps;         // bit i * k + j: tap (i, j) lies in the image (kernels of up to 32 taps)
    bool col;              // n < N

    __device__ __forceinline__ void init(const ConvDesc &cd, int n, int N) {
        col = n < N;
        const int ho = col ? n / cd.wcol : 0, wo = col ? n - ho * cd.wcol : 0;
        h0 = ho * cd.stride - cd.pad;
        w0 = wo * cd.stride - cd.pad;
        base = h0 * cd.W + w0;
        taps = 0;
        if (cd.kk <= 32)
            for (int i = 0, r = 0; i < cd.k; ++i)
                for (int j = 0; j < cd.k; ++j, ++r)
                    taps |= (inside(cd, i, j) ? 1u : 0u) << r;
    }
    __device__ __forceinline__ bool inside(const ConvDesc &cd, int i, int j) const {
        return col && (unsigned)(h0 + i) < (unsigned)cd.H && (unsigned)(w0 + j) < (unsigned)cd.W;
    }

    // Rows k0 .. of K.  k's channel and tap come from two multiplications on
    // the scalar unit (a table of offsets put its load's latency in front of
    // every step's gather), the bounds from the tap's bit, and an element
    // outside reads a zero instead of waiting for its value to be masked: four
    // vector instructions an element next to its load.
    __device__ __forceinline__ void load(const ConvDesc &cd, int k0, int K, int t) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int kl = __builtin_amdgcn_readfirstlane(k0 + t / BN + e * KSTEP), k = kl + cd.k0;
            const int c = (int)(((unsigned long long)(unsigned)k * cd.m_kk) >> cd.s_kk), r = k - c * cd.kk;
            const int i = (int)(((unsigned long long)(unsigned)r * cd.m_k) >> cd.s_k), j = r - i * cd.k;
            bool in;
            if (cd.kk <= 32) in = (taps & (kl < K ? 1u << r : 0u)) != 0;
            else in = kl < K && inside(cd, i, j);
            const float *p = cd.in + (unsigned)(base + c * (cd.H * cd.W) + i * cd.W + j);
            v[e] = *(in ? p : &kConvZero);
        }
    }

    // L[k][n], row length LD.
    template <int LD>
    __device__ __forceinline__ void store(float *L, int t) const {
#pragma unroll
        for (int e = 0; e < NE; ++e) L[(t / BN + e * KSTEP) * LD + t % BN] = v[e];
    }
};

template <bool CONV, int BK, int BN, int NT>
struct ConvRegsOf {
    typedef ConvRegs<BK, BN, NT> type;
};
template <int BK, int BN, int NT>
struct ConvRegsOf<false, BK, BN, NT> {
    typedef int type;
};

}  // namespace
}  // namespace ugemm
