// Split-form GEMM of small grids in one launch: no planes, no workspace.
//
// The plane-streaming path (gemm_mfma.hip) runs a preparation launch or more,
// FP16X3 a fill and a row-maximum pass first, then the core: on a problem of a
// few tiles each of them costs its launch, 4-5 us, and the core's one wave a
// SIMD a serial chain of K steps.  Here a workgroup of KG waves computes one
// (16 FM) x (16 FN) tile of C, wave w the 32-deep K steps w, w + KG, ...: a lane
// loads its fragment's eight FP32 values straight from the operand in either
// layout (two 16-byte loads of a k-contiguous one, eight 4-byte loads of a
// row-contiguous one, 16 lanes to 64 contiguous bytes), splits them in
// registers and feeds the MFMAs, with the next step's loads in flight.  The
// waves' sums are added through LDS in wave order, so calls are repeatable.
// FP16X3 runs over K twice: once for the row maxima of its panels, then, from
// the caches, for the products; every panel is scanned and split by each tile
// that needs it, which is what bounds the grids this pays for.
//
// The operands' splits, scales and products are those of the core; only the
// order of the FP32 sum differs (shorter partial sums).
#include "internal.h"
#include "kernel_common.h"
#include "split_common.h"

namespace ugemm {
namespace {

// Eight values k .. k+7 of row `row` of an operand of `rows` rows (KC:
// X[row*ld + k], else X[k*ld + row]).  Rows past the last read the last (their
// products are not stored); TAIL: K may end inside, values past it are 0.
template <bool KC, bool TAIL>
__device__ __forceinline__ void load_frag(const float *__restrict__ X, long ld, int rows, int row, int k, int K,
                                          float (&v)[8]) {
    row = min(row, rows - 1);
    if constexpr (TAIL) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int kj = min(k + j, K - 1);
            const float x = KC ? X[(long)row * ld + kj] : X[(long)kj * ld + row];
            v[j] = k + j < K ? x : 0.0f;
        }
    } else if constexpr (KC) {
        const float *p = X + (long)row * ld + k;
        const f32x4u a = *reinterpret_cast<const f32x4u *>(p), b = *reinterpret_cast<const f32x4u *>(p + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = a[j];
            v[4 + j] = b[j];
        }
    } else {
        const float *p = X + (long)k * ld + row;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[j * ld];
    }
}

template <int NP, class FMT, bool KCA, bool KCB, int FM, int FN, int KG>
__global__ __launch_bounds__(64 * KG) void split_small_kernel(int M, int N, int K, float alpha,
                                                              const float *__restrict__ A, long lda,
                                                              const float *__restrict__ B, long ldb, float beta,
                                                              float *__restrict__ C, long ldc, int tiles_m, int tiles_n,
                                                              Epilogue epi) {
    using V8 = typename FMT::V8;
    constexpr int BM = 16 * FM, BN = 16 * FN, LD = BN + 4, NT = 64 * KG;   // LD: conflict-free fragment stores
    __shared__ float red[KG][BM * LD];
    __shared__ unsigned smax[BM + BN];   // scaled formats: row maxima of the panels
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    const int steps = (K + 31) / 32;

    float ra[FM][8], rb[FN][8];
    auto load = [&](int s) {
        const int k = s * 32 + fk;
        if (s * 32 + 32 <= K) {
#pragma unroll
            for (int i = 0; i < FM; ++i) load_frag<KCA, false>(A, lda, M, m0 + i * 16 + fr, k, K, ra[i]);
#pragma unroll
            for (int j = 0; j < FN; ++j) load_frag<KCB, false>(B, ldb, N, n0 + j * 16 + fr, k, K, rb[j]);
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i) load_frag<KCA, true>(A, lda, M, m0 + i * 16 + fr, k, K, ra[i]);
#pragma unroll
            for (int j = 0; j < FN; ++j) load_frag<KCB, true>(B, ldb, N, n0 + j * 16 + fr, k, K, rb[j]);
        }
    };

    int ea[FM], eb[FN];     // scaled formats: exponents to add
    bool row_inf = false;   // and whether a row's largest magnitude is infinite
    const int mine = w < steps ? (steps - 1 - w) / KG + 1 : 0;   // this wave's steps: w + KG * u, u < mine
    if constexpr (FMT::SCALED) {
        if (t < BM + BN) smax[t] = 0u;
        float ma[FM], mb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) ma[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < FN; ++j) mb[j] = 0.0f;
        // Last step first: the products then start on step 0's values in hand.
        for (int u = mine - 1; u >= 0; --u) {
            load(w + KG * u);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
#pragma unroll
                for (int i = 0; i < FM; ++i) ma[i] = fmaxf(ma[i], fabsf(ra[i][q]));
#pragma unroll
                for (int j = 0; j < FN; ++j) mb[j] = fmaxf(mb[j], fabsf(rb[j][q]));
            }
        }
        __syncthreads();   // smax is zero
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            float m = fmaxf(ma[i], __shfl_xor(ma[i], 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            if (lane < 16 && m > 0.0f) atomicMax(&smax[i * 16 + fr], __float_as_uint(m));
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            float m = fmaxf(mb[j], __shfl_xor(mb[j], 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            if (lane < 16 && m > 0.0f) atomicMax(&smax[BM + j * 16 + fr], __float_as_uint(m));
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            ea[i] = -row_exp(smax[i * 16 + fr]);
            row_inf |= row_is_inf(smax[i * 16 + fr]);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            eb[j] = -row_exp(smax[BM + j * 16 + fr]);
            row_inf |= row_is_inf(smax[BM + j * 16 + fr]);
        }
        row_inf = __any(row_inf);
    } else if (mine > 0) {
        load(w);
    }

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int u = 0; u < mine; ++u) {
        // One answer for all fragments: a branch for the step.  Three planes
        // have no registers for both ways (spilling, 700x700x700 TT took 28.6
        // us instead of 17.8).
        bool special = NP == 3 || (FMT::SCALED && row_inf);
        if constexpr (!FMT::SCALED && NP == 2) {
#pragma unroll
            for (int i = 0; i < FM; ++i) special |= split_special(FMT(), ra[i], false);
#pragma unroll
            for (int j = 0; j < FN; ++j) special |= split_special(FMT(), rb[j], false);
            special = __any(special);
        }
        V8 pa[FM][NP], pb[FN][NP];
        auto split = [&](float (&x)[8], int e, bool sp, V8 (&w)[NP]) {
            if constexpr (FMT::SCALED) {
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] = ldexpf(x[q], e);
            }
            split8<NP, FMT>(x, sp, w);
        };
        auto split_all = [&](bool sp) {
#pragma unroll
            for (int i = 0; i < FM; ++i) split(ra[i], FMT::SCALED ? ea[i] : 0, sp, pa[i]);
#pragma unroll
            for (int j = 0; j < FN; ++j) split(rb[j], FMT::SCALED ? eb[j] : 0, sp, pb[j]);
        };
        if (special) split_all(true);
        else split_all(false);
        if (u + 1 < mine) load(w + KG * (u + 1));
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front of the MFMAs
#pragma unroll
        for (int q = 0; q < Products<NP>::N; ++q)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = FMT::mfma(pa[i][Products<NP>::a[q]], pb[j][Products<NP>::b[q]], acc[i][j]);
    }

    // Every wave's sums into LDS, then one value per thread and turn.
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[w][(i * 16 + (lane >> 4) * 4 + r) * LD + j * 16 + fr] = acc[i][j][r];
    __syncthreads();
    const bool has_epi = epi.active();
    static_assert(BM * BN % NT == 0, "whole turns");
#pragma unroll 2
    for (int e = t; e < BM * BN; e += NT) {
        const int r = e / BN, c = e % BN, m = m0 + r, n = n0 + c;
        if (m >= M || n >= N) continue;
        float x = red[0][r * LD + c];
#pragma unroll
        for (int h = 1; h < KG; ++h) x += red[h][r * LD + c];
        if constexpr (FMT::SCALED) x = ldexpf(x, row_exp(smax[r]) + row_exp(smax[BM + c]));
        float *cp = C + (long)m * ldc + n;
        float v = beta == 0.0f ? alpha * x : fmaf(alpha, x, beta * *cp);
        if (has_epi) v = apply_epilogue(epi, v, m, n);
        *cp = v;
    }
}

template <int NP, class FMT, int FM, int FN, int KG>
int launch(const Gemm<float> &g, hipStream_t s) {
    const int tiles_m = (g.M + 16 * FM - 1) / (16 * FM), tiles_n = (g.N + 16 * FN - 1) / (16 * FN);
    const dim3 grid((unsigned)(tiles_m * tiles_n)), block(64 * KG);
    timing_begin(s);
#define UGEMM_L(KCA, KCB)                                                                                              \
    hipLaunchKernelGGL((split_small_kernel<NP, FMT, KCA, KCB, FM, FN, KG>), grid, block, 0, s, g.M, g.N, g.K, g.alpha, \
                       g.A, g.lda, g.B, g.ldb, g.beta, g.C, g.ldc, tiles_m, tiles_n, g.epi)
    if (!g.ta && !g.tb) UGEMM_L(true, false);
    else if (!g.ta && g.tb) UGEMM_L(true, true);
    else if (g.ta && !g.tb) UGEMM_L(false, false);
    else UGEMM_L(false, true);
#undef UGEMM_L
    timing_end(s);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? UGEMM_OK : hip_fail(e, "small split launch");
}

template <int NP, class FMT = FmtBf16>
int launch_np(const Gemm<float> &g, int tile, hipStream_t s) {
    return tile == 32 ? launch<NP, FMT, 2, 2, 16>(g, s) : launch<NP, FMT, 4, 4, 8>(g, s);
}

}  // namespace

// us a call, planes / 32x32x16 waves / 64x64x8 waves (FP16X3; BF16X3):
//   512x512x512 (256 tiles of 32x32) 25.7 / 8.8 / 19.0;  16.4 / 6.9 / 14.9
//   700x700x700 (484) 33.6 / 22.0 / 25.2;  22.1 / 14.8 / 19.0
//   35x5120x1876 TN (320) 63 / 42 / 48;  31 / 24 / 30
//   832x64x1728 (52) 33.3 / 20.1 / 46.6;  21.7 / 13.2 / 32.0
//   543x128x3603 TT (68) 47.5 / 44.6 / 90;  25.9 / 32.6 / 64
//   1024x1024x1024 (256 of 64x64) 35.2 / 44.8 / 33.0;  27.0 / 30.3 / 23.1
//   5888x110x24 NT (184 of 64x64) 26.6 / 13.6 / 10.0;  10.2 / 10.2 / 8.5
//   1400x1400x300 (484 of 64x64) 28.3 / 54 / 27.8;  17.1 / 28.8 / 22.9
//   1615x2637x35 TN (1092 of 64x64) 37.2 / 71 / 31.9;  15.9 / 36.8 / 25.7
// So 32x32 tiles up to two workgroups a CU while the scan of K is short, 64x64
// up to one; FP16X3, whose planes cost three more launches, further where K
// is short.  A no-allocation call whose planes exceed the static scratch keeps
// the planes, and is refused as ever.
int split_small_tile(const Gemm<float> &g, int mode) {
    if (stream_alloc_is_static() && !mfma_planes_fit_scratch(g, mode)) return 0;
    const bool scaled = mode == UGEMM_MODE_FP16X3;
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (t32 <= 2 * cus && g.K <= (scaled && t32 <= cus ? 3072 : 2048)) return 32;
    if (t64 <= cus && g.K <= 1024) return 64;
    return scaled && ((t64 <= 2 * cus && g.K <= 256) || (t64 <= 4 * cus && g.K <= 64)) ? 64 : 0;
}

int launch_split_small(const Gemm<float> &g, int mode, int tile, hipStream_t s) {
    switch (mode) {
        case UGEMM_MODE_BF16X1: return launch_np<1>(g, tile, s);
        case UGEMM_MODE_BF16X3: return launch_np<2>(g, tile, s);
        case UGEMM_MODE_BF16X6: return launch_np<3>(g, tile, s);
        case UGEMM_MODE_FP16X3: return launch_np<2, FmtF16>(g, tile, s);
        default: return fail(UGEMM_ERR_UNSUPPORTED, "mode %d is not a split form", mode);
    }
}

}  // namespace ugemm
