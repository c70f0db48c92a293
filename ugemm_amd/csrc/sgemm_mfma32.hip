// FP32 SGEMM on the FP32 matrix cores of gfx950 (v_mfma_f32_16x16x4_f32):
// FP32 operands as given, FP32 products, FP32 accumulation -- no operand
// split or conversion, so no preparation kernels and the error class of the
// plain FP32 kernel.  MI355X's FP32 MFMA peak (157.3 TF/s) equals its FP32
// vector peak, but the matrix core is fed one register per operand per 2048
// flop instead of one per 2 flop, so it runs much closer to that peak.
// The tile computation (LDS layout, k-permuted fragments) is m32_tile in
// mfma32_tile.h.
//
// Split-K (gridDim.y > 1): block (tile, z) multiplies K columns
// [z*kc, min(K, (z+1)*kc)) into the partial slice ws + z*M*N; the partials
// are added in fixed order by the split-K reduction, which also applies
// alpha, beta and the epilogue.  Repeated calls are bitwise identical.
#include <algorithm>

#include "internal.h"
#include "kernel_common.h"
#include "mfma32_tile.h"

namespace ugemm {
namespace {

template <class CF, bool TA, bool TB>
__global__ __launch_bounds__(CF::THREADS, CF::MINB) void sgemm_mfma32_kernel(
    int M, int N, int K_, float alpha_, const float *__restrict__ A_, long lda, const float *__restrict__ B_,
    long ldb, float beta_, float *__restrict__ C_, long ldc_, int tiles_m, int tiles_n, Epilogue epi, int kc,
    float *__restrict__ ws) {
    // This layout's two stages of both operands (at most CF::kLdsFloats).
    __shared__ __attribute__((aligned(16))) float lds[CF::template lds_floats<TA, TB>()];
    const bool part = gridDim.y > 1;
    const int kz0 = part ? (int)blockIdx.y * kc : 0;
    const int K = part ? min(kc, K_ - kz0) : K_;
    const float *A = TA ? A_ + (long)kz0 * lda : A_ + kz0;
    const float *B = TB ? B_ + kz0 : B_ + (long)kz0 * ldb;
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    m32_tile<CF, TA, TB>(M, N, K, part ? 1.0f : alpha_, A, lda, B, ldb, part ? 0.0f : beta_,
                         part ? ws + (long)blockIdx.y * M * N : C_, part ? (long)N : ldc_, tm * CF::BM, tn * CF::BN, lds,
                         part ? Epilogue() : epi);
}

// Implicit-GEMM convolution on the FP32 matrix cores: C (M = output
// channels x N = output pixels) = W (M x K, row-major weights) * im2col(in),
// then the epilogue; the column matrix is gathered in the tile loader
// (ConvDesc).  Split-K as in the GEMM kernel: the chunk's weight columns, and
// cd.k0, from which its k count (ConvRegs).
template <class CF>
__global__ __launch_bounds__(CF::THREADS, CF::MINB) void conv_mfma32_kernel(
    int M, int N, int K_, const float *__restrict__ A_, long lda, float *__restrict__ C_, long ldc_, int tiles_m,
    int tiles_n, Epilogue epi, ConvDesc cd, int kc, float *__restrict__ ws) {
    __shared__ __attribute__((aligned(16))) float lds[CF::template lds_floats<false, false>()];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const bool part = gridDim.y > 1;
    const int k0 = part ? (int)blockIdx.y * kc : 0;
    ConvDesc cz = cd;
    cz.k0 = k0;
    m32_tile<CF, false, false, true>(M, N, part ? min(kc, K_ - k0) : K_, 1.0f, A_ + k0, lda, nullptr, 0, 0.0f,
                                     part ? ws + (long)blockIdx.y * M * N : C_, part ? (long)N : ldc_, tm * CF::BM,
                                     tn * CF::BN, lds, part ? Epilogue() : epi, cz);
}

using V0 = M32Cfg<128, 128, 16, 2, 2, 2>;
using V1 = M32Cfg<256, 128, 16, 4, 2>;
using V2 = M32Cfg<128, 256, 16, 2, 4>;
using V3 = M32Cfg<64, 64, 16, 2, 2, 2>;
using V4 = M32Cfg<256, 256, 16, 2, 4>;
using V5 = M32Cfg<128, 128, 32, 2, 2, 2>;
// Small grids (launch_small): K dealt to groups of one workgroup.
using V3K4 = M32Cfg<64, 64, 16, 2, 2, 1, 4>;
using V3S8 = M32Cfg<32, 32, 16, 1, 1, 1, 8>;
using V3S16 = M32Cfg<32, 32, 16, 1, 1, 1, 16>;
using V3C8 = M32Cfg<32, 64, 16, 1, 2, 1, 8>;   // convolutions

const char *kNames[] = {"f32_mfma_128x128x16_w2x2", "f32_mfma_256x128x16_w4x2", "f32_mfma_128x256x16_w2x4",
                        "f32_mfma_64x64x16_w2x2",   "f32_mfma_256x256x16_w2x4", "f32_mfma_128x128x32_w2x2"};
constexpr int kNum = 6;

template <class CF>
int launch_cfg(const Gemm<float> &g, hipStream_t s) {
    const int tiles_m = (g.M + CF::BM - 1) / CF::BM, tiles_n = (g.N + CF::BN - 1) / CF::BN;
    const long nblk = (long)tiles_m * tiles_n;
    if (nblk > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "sgemm fp32 mfma: too many tiles (%ld)", nblk);
    int kc = g.K;
    const int splits = split_count(g.splits, nblk, g.K, 64, &kc, 2);
    float *ws = nullptr;
    if (splits > 1) {
        const int rc = stream_alloc((void **)&ws, (size_t)splits * g.M * g.N * sizeof(float), s);
        if (rc) return rc;
    }
    dim3 grid((unsigned)nblk, (unsigned)splits), block(CF::THREADS);
#define UGEMM_L(TA, TB) \
    hipLaunchKernelGGL((sgemm_mfma32_kernel<CF, TA, TB>), grid, block, 0, s, g.M, g.N, g.K, g.alpha, g.A, \
                       g.lda, g.B, g.ldb, g.beta, g.C, g.ldc, tiles_m, tiles_n, g.epi, kc, ws)
    timing_begin(s);
    if (!g.ta && !g.tb) UGEMM_L(false, false);
    else if (!g.ta && g.tb) UGEMM_L(false, true);
    else if (g.ta && !g.tb) UGEMM_L(true, false);
    else UGEMM_L(true, true);
    timing_end(s);
#undef UGEMM_L
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "sgemm fp32 mfma launch");
    if (splits > 1) {
        if (!rc) rc = launch_splitk_reduce_f32(g.M, g.N, splits, g.alpha, ws, g.beta, g.C, g.ldc, g.epi, s);
        const int rc2 = stream_free(ws, s);
        if (!rc) rc = rc2;
    }
    return rc;
}

// Variant 3 with the automatic split count: K dealt to groups of a workgroup
// where the grid leaves a CU one wave a SIMD (the reasons stand at the FP32
// kernel's launch_small).  us a call, 64x64x1 / 64x64x4 / 32x32x8 / 32x32x16:
//   128x96x200 14.2 / 10.4 / 6.8 / 7.1;  512x512x512 18.8 / 15.8 / 8.6 / 8.9;  28x768x1472 65 / 41 / 18 / 17;
//   700x700x2000 115 / 54 / 36 / 37;  1023x1000x1023 61 / 31 / 38 / 46;  2720x1313x87 17.1 / 18.7 / 30 / 52.
int launch_small(const Gemm<float> &g, hipStream_t s) {
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (g.splits != 0 || t64 > 4 * cus) return launch_cfg<V3>(g, s);
    Gemm<float> h = g;
    h.splits = 1;
    if (t32 <= cus && t32 * g.K <= cus * 4096) {
        if (g.K > 1024) h.splits = (int)std::max(1L, std::min({cus / t32, g.K / 384L, 16L}));
        return launch_cfg<V3S16>(h, s);
    }
    if (t32 <= 2 * cus && g.K <= 2048) return launch_cfg<V3S8>(h, s);
    // One tile a CU and a K of a few steps: a chain of latencies that deal_k,
    // fitted to longer ones, prices too low (us, one group / four: 4440x192x128
    // 11.1 / 8.8, 1000x1000x200 15.3 / 11.3, 4440x192x256 16.5 / 11.9, K 64 8.5 / 8.5).
    if (t64 <= cus && g.K > 64 && g.K <= 512) return launch_cfg<V3K4>(h, s);
    return deal_k(t64, g.K, 21.0, 2, sizeof(*g.C) * g.M * g.N, &h.splits) ? (h.splits = 1, launch_cfg<V3K4>(h, s)) : launch_cfg<V3>(h, s);
}

template <class CF>
int launch_conv_cfg(const Gemm<float> &g, const ConvDesc &cd, hipStream_t s) {
    const int tiles_m = (g.M + CF::BM - 1) / CF::BM, tiles_n = (g.N + CF::BN - 1) / CF::BN;
    const long nblk = (long)tiles_m * tiles_n;
    if (nblk > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "conv fp32 mfma: too many tiles (%ld)", nblk);
    int kc = g.K;
    const int splits = split_count(g.splits, nblk, g.K, 64, &kc, 2);
    float *ws = nullptr;
    if (splits > 1) {
        const int rc = stream_alloc((void **)&ws, (size_t)splits * g.M * g.N * sizeof(float), s);
        if (rc) return rc;
    }
    timing_begin(s);
    hipLaunchKernelGGL((conv_mfma32_kernel<CF>), dim3((unsigned)nblk, (unsigned)splits), dim3(CF::THREADS), 0, s, g.M,
                       g.N, g.K, g.A, g.lda, g.C, g.ldc, tiles_m, tiles_n, g.epi, cd, kc, ws);
    timing_end(s);
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "conv fp32 mfma launch");
    if (splits > 1) {
        if (!rc) rc = launch_splitk_reduce_f32(g.M, g.N, splits, 1.0f, ws, 0.0f, g.C, g.ldc, g.epi, s);
        const int rc2 = stream_free(ws, s);
        if (!rc) rc = rc2;
    }
    return rc;
}

// Variant 3 with the automatic split count, as the FP32 kernel's.
int launch_conv_small(const Gemm<float> &g, const ConvDesc &cd, hipStream_t s) {
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 63) / 64), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (g.splits != 0 || t64 > 4 * cus) return launch_conv_cfg<V3>(g, cd, s);
    Gemm<float> h = g;
    h.splits = 1;
    if (t32 <= cus && t32 * g.K <= cus * 2048) {
        if (g.K > 768) h.splits = (int)std::max(1L, std::min({cus / t32, g.K / 256L, 16L}));
        return launch_conv_cfg<V3C8>(h, cd, s);
    }
    return deal_k(t64, g.K, 40.0, 2, sizeof(*g.C) * g.M * g.N, &h.splits) ? (h.splits = 1, launch_conv_cfg<V3K4>(h, cd, s))
                                                                        : launch_conv_cfg<V3>(h, cd, s);
}

}  // namespace

int m32_variant_count() { return kNum; }
const char *m32_variant_name(int v) { return (v >= 0 && v < kNum) ? kNames[v] : nullptr; }

// 256x128 tiles of 8 waves wherever they fill every CU (measured on MI355X at
// 8192^3 NN: 137 TF/s against 122 for 128x128, and 131 against 106 on
// 65536x256x4096); 128x128 when those fill it; 64x64 below (with split-K
// on a grid that is still short).
int m32_pick_variant(const Gemm<float> &g) {
    const long cus = device_cu_count();
    const long t256 = (long)((g.M + 255) / 256) * ((g.N + 127) / 128);
    const long t128 = (long)((g.M + 127) / 128) * ((g.N + 127) / 128);
    const int v = t256 >= cus ? 1 : t128 >= cus ? 0 : 3;
    if (t128 <= cus) return v;
    // As fp32_pick_variant, over the same 60 sizes: 1.19 times as fast on
    // average as by the count of 256x128 tiles alone.
    static const TileCost cost[4] = {{128, 128, 62, 0.47}, {256, 128, 58.5, 0.3}, {128, 256, 58.5, 0.3}, {64, 64, 70, 1.1}};
    return cheapest_tile(cost, 4, 0, v, g.M, g.N);
}

// g: the convolution as a GEMM (alpha 1, beta 0, A the weights, B unused).
int launch_conv_m32(const Gemm<float> &g, const ConvDesc &cd, int variant, hipStream_t s) {
    if (variant < 0) variant = 3;   // the fastest at every size tried: the gather sets the pace
    switch (variant) {
        case 0: return launch_conv_cfg<V0>(g, cd, s);
        case 1: return launch_conv_cfg<V1>(g, cd, s);
        case 2: return launch_conv_cfg<V2>(g, cd, s);
        case 3: return launch_conv_small(g, cd, s);
        case 4: return launch_conv_cfg<V4>(g, cd, s);
        case 5: return launch_conv_cfg<V5>(g, cd, s);
        default: return fail(UGEMM_ERR_ARG, "conv fp32 mfma: no variant %d", variant);
    }
}

int launch_m32(const Gemm<float> &g, int variant, hipStream_t s) {
    switch (variant) {
        case 0: return launch_cfg<V0>(g, s);
        case 1: return launch_cfg<V1>(g, s);
        case 2: return launch_cfg<V2>(g, s);
        case 3: return launch_small(g, s);
        case 4: return launch_cfg<V4>(g, s);
        case 5: return launch_cfg<V5>(g, s);
        default: return fail(UGEMM_ERR_ARG, "sgemm fp32 mfma: no variant %d", variant);
    }
}

}  // namespace ugemm
