// Plain FP32 SGEMM for gfx950: vector FMA with FP32 accumulation, one
// workgroup per C tile (tile body in fp32_tile.h).  Tiles are visited in the
// XCD-aware order of tile_coords (kernel_common.h).
#include <algorithm>

#include "internal.h"
#include "fp32_tile.h"

namespace ugemm {
namespace {

// Split-K (gridDim.y > 1): block (tile, z) multiplies K columns
// [z*kc, min(K, (z+1)*kc)) into the partial slice ws + z*M*N (row length N).
template <class CF, bool TA, bool TB>
__global__ __launch_bounds__(CF::THREADS, CF::MINB) void sgemm_fp32_kernel(int M, int N, int K, float alpha,
                                                            const float *__restrict__ A, long lda,
                                                            const float *__restrict__ B, long ldb, float beta,
                                                            float *__restrict__ C, long ldc, int tiles_m, int tiles_n,
                                                            Epilogue epi, int kc, float *__restrict__ ws) {
    __shared__ __attribute__((aligned(16))) float lds[CF::kLdsFloats];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const bool part = gridDim.y > 1;
    const int k0 = part ? (int)blockIdx.y * kc : 0;
    fp32_tile<CF, TA, TB>(M, N, part ? min(kc, K - k0) : K, part ? 1.0f : alpha, TA ? A + (long)k0 * lda : A + k0, lda,
                          TB ? B + k0 : B + (long)k0 * ldb, ldb, part ? 0.0f : beta,
                          part ? ws + (long)blockIdx.y * M * N : C, part ? (long)N : ldc, tm * CF::BM, tn * CF::BN, lds,
                          part ? Epilogue() : epi);
}

// Implicit-GEMM convolution: C (M = output channels x N = output pixels) =
// alpha * W (M x K, row-major weights) * im2col(in) + beta * C, then the
// epilogue.  The column matrix is gathered in the tile loader (ConvDesc).
// Split-K as in sgemm_fp32_kernel: the chunk's weight columns, and cd.k0, from
// which its k count (ConvRegs).
template <class CF>
__global__ __launch_bounds__(CF::THREADS) void conv_fp32_kernel(int M, int N, int K, float alpha,
                                                           const float *__restrict__ A, long lda, float beta,
                                                           float *__restrict__ C, long ldc, int tiles_m, int tiles_n,
                                                           Epilogue epi, ConvDesc cd, int kc, float *__restrict__ ws) {
    __shared__ __attribute__((aligned(16))) float lds[CF::kLdsFloats];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const bool part = gridDim.y > 1;
    const int k0 = part ? (int)blockIdx.y * kc : 0;
    ConvDesc cz = cd;
    cz.k0 = k0;
    fp32_tile<CF, false, false, true>(M, N, part ? min(kc, K - k0) : K, part ? 1.0f : alpha, A + k0, lda, nullptr, 0,
                                      part ? 0.0f : beta, part ? ws + (long)blockIdx.y * M * N : C,
                                      part ? (long)N : ldc, tm * CF::BM, tn * CF::BN, lds, part ? Epilogue() : epi, cz);
}

// ---------------------------------------------------------------------------
// Variant table.
using V0 = Fp32Cfg<128, 128, 16, 8, 8>;
using V1 = Fp32Cfg<64, 64, 16, 4, 4>;
using V2 = Fp32Cfg<128, 64, 16, 8, 4>;
using V3 = Fp32Cfg<64, 128, 16, 4, 8>;
using V4 = Fp32Cfg<256, 128, 16, 16, 8, 2>;
using V5 = Fp32Cfg<128, 256, 16, 8, 16, 2>;

// Small grids (launch_small): K dealt to groups of one workgroup.
using V1K4 = Fp32Cfg<64, 64, 16, 4, 4, 1, 4>;
using V1S8 = Fp32Cfg<32, 32, 16, 4, 4, 1, 8>;
using V1S16 = Fp32Cfg<32, 32, 16, 4, 4, 1, 16>;
using V1C8 = Fp32Cfg<32, 64, 16, 4, 4, 1, 8>;   // convolutions

const char *kNames[] = {"fp32_128x128x16_t8x8", "fp32_64x64x16_t4x4", "fp32_128x64x16_t8x4",
                        "fp32_64x128x16_t4x8", "fp32_256x128x16_t16x8", "fp32_128x256x16_t8x16"};
constexpr int kNumVariants = 6;

template <class CF>
int launch_cfg(const Gemm<float> &g, hipStream_t s) {
    const int tiles_m = (g.M + CF::BM - 1) / CF::BM;
    const int tiles_n = (g.N + CF::BN - 1) / CF::BN;
    const long nblk = (long)tiles_m * tiles_n;
    if (nblk > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "sgemm: too many tiles (%ld)", nblk);
    int kc = g.K;
    const int splits = split_count(g.splits, nblk, g.K, 64, &kc, 2);
    float *ws = nullptr;
    if (splits > 1) {
        const int rc = stream_alloc((void **)&ws, (size_t)splits * g.M * g.N * sizeof(float), s);
        if (rc) return rc;
    }
    dim3 grid((unsigned)nblk, (unsigned)splits), block(CF::THREADS);
#define UGEMM_L(TA, TB) \
    hipLaunchKernelGGL((sgemm_fp32_kernel<CF, TA, TB>), grid, block, 0, s, g.M, g.N, g.K, g.alpha, g.A, \
                       g.lda, g.B, g.ldb, g.beta, g.C, g.ldc, tiles_m, tiles_n, g.epi, kc, ws)
    timing_begin(s);
    if (!g.ta && !g.tb) UGEMM_L(false, false);
    else if (!g.ta && g.tb) UGEMM_L(false, true);
    else if (g.ta && !g.tb) UGEMM_L(true, false);
    else UGEMM_L(true, true);
    timing_end(s);
#undef UGEMM_L
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "sgemm launch");
    if (splits > 1) {
        if (!rc) rc = launch_splitk_reduce_f32(g.M, g.N, splits, g.alpha, ws, g.beta, g.C, g.ldc, g.epi, s);
        const int rc2 = stream_free(ws, s);
        if (!rc) rc = rc2;
    }
    return rc;
}

// Variant 1 with the automatic split count.  A grid of few tiles leaves a CU
// one wave a SIMD and a serial chain of K steps of 1.2 us each; K is then
// dealt to the groups of a workgroup instead of chunks and a second launch (5
// us on top of a 7 us call).  us a call by tile and groups, 64x64x1 / 64x64x4 / 32x32x8 / 32x32x16:
//   128x96x200 (12 tiles of 32x32) 17.5 / 10.9 / 6.8 / 6.9;  512x512x512 (256) 27.5 / 16.9 / 8.7 / 8.8;
//   28x768x1472 (24) 96 / 44 / 19.9 / 17.7;  700x700x2000 (484) 157 / 61 / 41.6 / 43.0;
//   1023x1000x1023 (1024; 256 of 64x64) 82 / 37 / 44 / 50;  1400x1400x300 (484 of 64x64) 26.0 / 23.9 / 31 / 47;
//   2720x1313x87 (903 of 64x64) 18.2 / 19.5 / 27 / 49.
// 32x32 tiles in groups of 8 or 16 serve the smallest grids (at 7 us per 1000
// of K; past 1024 the CUs that are left take chunks of it) while the product
// is short of 4096 of K on every CU; deal_k chooses for the others.
int launch_small(const Gemm<float> &g, hipStream_t s) {
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (g.splits != 0 || t64 > 4 * cus) return launch_cfg<V1>(g, s);
    Gemm<float> h = g;
    h.splits = 1;
    if (t32 <= cus && t32 * g.K <= cus * 4096) {
        if (g.K > 1024) h.splits = (int)std::max(1L, std::min({cus / t32, g.K / 384L, 16L}));
        return launch_cfg<V1S16>(h, s);
    }
    if (t32 <= 2 * cus && g.K <= 2048) return launch_cfg<V1S8>(h, s);
    return deal_k(t64, g.K, 28.0, 2, sizeof(*g.C) * g.M * g.N, &h.splits) ? (h.splits = 1, launch_cfg<V1K4>(h, s)) : launch_cfg<V1>(h, s);
}

template <class CF>
int launch_conv_cfg(const Gemm<float> &g, const ConvDesc &cd, hipStream_t s) {
    const int tiles_m = (g.M + CF::BM - 1) / CF::BM;
    const int tiles_n = (g.N + CF::BN - 1) / CF::BN;
    const long nblk = (long)tiles_m * tiles_n;
    if (nblk > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "conv: too many tiles (%ld)", nblk);
    int kc = g.K;
    const int splits = split_count(g.splits, nblk, g.K, 64, &kc, 2);
    float *ws = nullptr;
    if (splits > 1) {
        const int rc = stream_alloc((void **)&ws, (size_t)splits * g.M * g.N * sizeof(float), s);
        if (rc) return rc;
    }
    dim3 grid((unsigned)nblk, (unsigned)splits), block(CF::THREADS);
    timing_begin(s);
    hipLaunchKernelGGL((conv_fp32_kernel<CF>), grid, block, 0, s, g.M, g.N, g.K, g.alpha, g.A, g.lda, g.beta, g.C,
                       g.ldc, tiles_m, tiles_n, g.epi, cd, kc, ws);
    timing_end(s);
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "conv launch");
    if (splits > 1) {
        if (!rc) rc = launch_splitk_reduce_f32(g.M, g.N, splits, g.alpha, ws, g.beta, g.C, g.ldc, g.epi, s);
        const int rc2 = stream_free(ws, s);
        if (!rc) rc = rc2;
    }
    return rc;
}

// Variant 1 with the automatic split count, as launch_small: 8 groups of 32x64
// tiles for the smallest grids, else as deal_k has it.
int launch_conv_small(const Gemm<float> &g, const ConvDesc &cd, hipStream_t s) {
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 63) / 64), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (g.splits != 0 || t64 > 4 * cus) return launch_conv_cfg<V1>(g, cd, s);
    Gemm<float> h = g;
    h.splits = 1;
    if (t32 <= cus && t32 * g.K <= cus * 2048) {
        if (g.K > 768) h.splits = (int)std::max(1L, std::min({cus / t32, g.K / 256L, 16L}));
        return launch_conv_cfg<V1C8>(h, cd, s);
    }
    return deal_k(t64, g.K, 40.0, 2, sizeof(*g.C) * g.M * g.N, &h.splits) ? (h.splits = 1, launch_conv_cfg<V1K4>(h, cd, s))
                                                                        : launch_conv_cfg<V1>(h, cd, s);
}

}  // namespace

int fp32_variant_count() { return kNumVariants; }
const char *fp32_variant_name(int v) { return (v >= 0 && v < kNumVariants) ? kNames[v] : nullptr; }

int fp32_pick_variant(const Gemm<float> &g) {
    // Enough 128x256 tiles to give every CU two: the 8x16 micro-tile, whose
    // k-step reads 24 floats from LDS per 128 FMAs (8x8: 16 per 64), the LDS
    // bandwidth that bounds the 8x8 kernel (measured 6-8% faster at 8192^3).
    // Else enough 128x128 tiles: those; otherwise shrink the tile so that the
    // grid still covers the chip.
    // Row-major NN (A k-contiguous, B row-contiguous) runs best on the 16x8
    // micro-tile: 98-100 against 92-93 TF/s for 8x16 at 4096^3 and 8192^3,
    // interleaved on one box; NT and TN stay on 8x16 (within 1-3% of 8x8).
    // A grid of 128x256 tiles covering half the CUs still takes 8x16, the
    // launcher splitting K (2048^3: 77 against 74 TF/s on 64x64 tiles).
    const int cus = device_cu_count();
    const long t128x256 = (long)((g.M + 127) / 128) * ((g.N + 255) / 256);
    const long t256x128 = (long)((g.M + 255) / 256) * ((g.N + 127) / 128);
    const long t128 = (long)((g.M + 127) / 128) * ((g.N + 127) / 128);
    const bool nn = !g.ta && !g.tb;
    int v;
    if (nn && t256x128 >= 2L * cus) v = 4;
    else if (t128x256 >= 2L * cus) v = 5;
    else if (t128 >= 2L * cus) v = 0;
    else if (2 * t128x256 >= cus && g.K >= 1024 && g.splits != 1) return 5;
    else {
        const long t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
        v = t64 > 2L * cus && g.M >= 4 * g.N ? 2 : t64 > 2L * cus && g.N >= 4 * g.M ? 3 : 1;
    }
    if (t128 <= cus) return v;
    // The CU with one tile more than the others sets the time: 583 tiles of
    // 128x128 (6662x1408x2930 NT) are three on some CUs and two on most, 890 us,
    // where 1166 of 128x64 are five and four, 756.  So another shape where the
    // tiles of its fullest CU are 5% cheaper (us per 128x128 and 1000 of K, a
    // lone tile's latency in tiles; fitted to all six over 60 sizes).  Over those
    // sizes (sides 720..16384, K 256..5800) 1.11 times as fast on average.
    static const TileCost cost[6] = {{128, 128, 85, 0.27}, {64, 64, 95, 0.9},   {128, 64, 87, 0.75},
                                     {64, 128, 87, 0.75},  {256, 128, 82, 0.23}, {128, 256, 82, 0.2}};
    return cheapest_tile(cost, 6, 1 << (nn ? 5 : 4), v, g.M, g.N);
}

int launch_conv_fp32(const Gemm<float> &g, const ConvDesc &cd, int variant, hipStream_t s) {
    // Convolutions are compiled for the four 8x8-or-smaller tiles; 64x64 is the
    // fastest of them at every size tried (the gather, not the FMAs, sets the pace).
    if (variant < 0) variant = 1;
    if (variant >= 4) variant = 0;
    switch (variant) {
        case 0: return launch_conv_cfg<V0>(g, cd, s);
        case 1: return launch_conv_small(g, cd, s);
        case 2: return launch_conv_cfg<V2>(g, cd, s);
        case 3: return launch_conv_cfg<V3>(g, cd, s);
        default: return fail(UGEMM_ERR_ARG, "conv: no variant %d", variant);
    }
}

int launch_fp32(const Gemm<float> &g, int variant, hipStream_t s) {
    switch (variant) {
        case 0: return launch_cfg<V0>(g, s);
        case 1: return launch_small(g, s);
        case 2: return launch_cfg<V2>(g, s);
        case 3: return launch_cfg<V3>(g, s);
        case 4: return launch_cfg<V4>(g, s);
        case 5: return launch_cfg<V5>(g, s);
        default: return fail(UGEMM_ERR_ARG, "fp32: no variant %d", variant);
    }
}

}  // namespace ugemm
