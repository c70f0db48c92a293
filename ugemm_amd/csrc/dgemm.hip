// DGEMM for gfx950 on FP64 MFMA (v_mfma_f64_16x16x4_f64), FP64 accumulation.
//
// One workgroup computes a BM x BN tile of C with 4 waves (2 x 2); each wave
// owns a (BM/2) x (BN/2) grid of 16x16 fragments.  Operand tiles of BK = 16
// move global -> registers -> LDS with the layout-aware loader shared with
// the FP32 kernel (transposed layouts are turned around while writing LDS),
// two LDS stages, one barrier per BK step.  LDS holds both operands K-major
// (As[k][m], Bs[k][n]) so that a fragment read -- lane l takes row l%16 of
// k-slice l/16 -- is one conflict-free ds_read_b64 over 128 contiguous bytes
// per 16 lanes.  The D fragment of the FP64 MFMA holds rows l/16 + 4*i,
// column l%16 (measured on gfx950: unlike the FP32-output forms, whose rows
// are 4*(l/16) + i).
//
// Determinism: every element of C is a fixed sequence of MFMAs over k, and a
// split-K call adds its partial slices in a fixed order (no atomics), so
// repeated calls are bitwise identical.
// Semantics as dgemm_cpu (ugemm.h:162-286) with the BLAS beta == 0 rule.
#include <algorithm>
#include <type_traits>

#include "internal.h"
#include "kernel_common.h"

namespace ugemm {
namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

// WG x WG waves to a tile.  KG: groups of them in a workgroup, each with its
// own LDS stages; group g multiplies K tiles g, g + KG, ... and the groups'
// sums are added through LDS in group order (small grids, launch_small).
// WEU: waves per SIMD the kernel is compiled for.
template <int BM_, int BN_, int WG_ = 2, int KG_ = 1, int WEU_ = 2>
struct DCfg {
    static constexpr int BM = BM_, BN = BN_, BK = 16, WG = WG_, NT = 64 * WG * WG, KG = KG_, WEU = WEU_;
    static constexpr int WTM = BM / WG, WTN = BN / WG, FM = WTM / 16, FN = WTN / 16;
    static constexpr int LDA = BM + 2, LDB = BN + 2;   // doubles; +2 keeps 16-byte alignment
    static constexpr int kStage = 2 * BK * (LDA + LDB);   // doubles: two stages of a group
    static_assert(KG == 1 || BM * BN <= kStage, "the groups' sums fit their stages");
};

// Split-K (gridDim.y > 1): block (tile, z) multiplies K columns
// [z*kc, min(K, (z+1)*kc)) into the partial slice ws + z*M*N (row length N).
template <class CF, bool TA, bool TB>
__global__ __launch_bounds__(CF::NT * CF::KG) __attribute__((amdgpu_waves_per_eu(CF::WEU))) void dgemm_mfma_kernel(
    int M, int N, int K_, double alpha_, const double *__restrict__ A_, long lda, const double *__restrict__ B_,
    long ldb, double beta_, double *__restrict__ C_, long ldc_, int tiles_m, int tiles_n, int kc,
    double *__restrict__ ws) {
    const bool part = gridDim.y > 1;
    const int kz0 = part ? (int)blockIdx.y * kc : 0;
    const int K = part ? min(kc, K_ - kz0) : K_;
    const double *__restrict__ A = TA ? A_ + (long)kz0 * lda : A_ + kz0;
    const double *__restrict__ B = TB ? B_ + kz0 : B_ + (long)kz0 * ldb;
    double *__restrict__ C = part ? ws + (long)blockIdx.y * M * N : C_;
    const long ldc = part ? (long)N : ldc_;
    const double alpha = part ? 1.0 : alpha_, beta = part ? 0.0 : beta_;
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, NT = CF::NT, FM = CF::FM, FN = CF::FN;
    constexpr int LDA = CF::LDA, LDB = CF::LDB;
    constexpr int KG = CF::KG;
    __shared__ __attribute__((aligned(16))) double lds[KG * CF::kStage];
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    double *As = lds + grp * CF::kStage, *Bs = As + 2 * BK * LDA;

    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int t = KG == 1 ? threadIdx.x : threadIdx.x % NT, lane = t & 63, w = t >> 6;
    const int wm = w / CF::WG, wn = w % CF::WG;

    using ARegs = TileRegs<double, TA ? BM : BK, TA ? BK : BM, NT>;
    using BRegs = TileRegs<double, TB ? BK : BN, TB ? BN : BK, NT>;
    ARegs ra;
    BRegs rb;
    const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
    const bool wide_a = (TA ? M : K) >= 2, wide_b = (TB ? K : N) >= 2;
    const int ktiles = (K + BK - 1) / BK, kfull = K / BK;

    // EDGE tiles reach past M, N or K.
    auto load_tile = [&](int kt, auto edge) {
        const int k0 = kt * BK;
        const double *a0 = TA ? A + (long)k0 * lda + m0 : A + (long)m0 * lda + k0;
        const double *b0 = TB ? B + (long)n0 * ldb + k0 : B + (long)k0 * ldb + n0;
        if constexpr (!decltype(edge)::value) {
            ra.load(a0, lda, t);
            rb.load(b0, ldb, t);
        } else {
            const int mr = M - m0, nr = N - n0, kr = K - k0;
            ra.load_edge(a0, lda, t, TA ? mr : kr, TA ? kr : mr, wide_a);
            rb.load_edge(b0, ldb, t, TB ? kr : nr, TB ? nr : kr, wide_b);
        }
    };
    auto store_tile = [&](int kt, int buf, auto edge) {
        if constexpr (decltype(edge)::value) {
            const int mr = M - m0, nr = N - n0, kr = K - kt * BK;
            ra.mask(t, TA ? mr : kr, TA ? kr : mr, wide_a);
            rb.mask(t, TB ? kr : nr, TB ? nr : kr, wide_b);
        }
        ra.template store<TA, LDA>(As + buf * BK * LDA, t);
        rb.template store<!TB, LDB>(Bs + buf * BK * LDB, t);
    };

    doublex4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = doublex4{0.0, 0.0, 0.0, 0.0};

    // K tiles below nfast are loaded without bounds; the others (all of an
    // edge tile's, and a K remainder) as edges, in a loop of their own.
    const int nfast = interior ? kfull : 0;
    if (grp < nfast) {
        load_tile(grp, std::false_type());
        store_tile(grp, 0, std::false_type());
    } else if (grp < ktiles) {
        load_tile(grp, std::true_type());
        store_tile(grp, 0, std::true_type());
    }
    __syncthreads();

    const int frow = lane & 15, fk = lane >> 4;
    auto step = [&](int kt, int buf, bool more, auto edge) {   // edge: of the group's next K tile
        if (more) load_tile(kt + KG, edge);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front of the multiplications
        const double *as = As + buf * BK * LDA + fk * LDA + wm * CF::WTM + frow;
        const double *bs = Bs + buf * BK * LDB + fk * LDB + wn * CF::WTN + frow;
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) {
            double fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[i] = as[s * 4 * LDA + i * 16];
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[j] = bs[s * 4 * LDB + j * 16];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) store_tile(kt + KG, buf ^ 1, edge);
        __syncthreads();
    };
    int kt = grp, buf = 0;
    for (; kt + KG < nfast; kt += KG, buf ^= 1) step(kt, buf, true, std::false_type());
    for (; kt < ktiles; kt += KG, buf ^= 1) step(kt, buf, kt + KG < ktiles, std::true_type());
    if constexpr (KG > 1) {
        // Groups with one K tile less join the last step's barrier.
        if (ktiles % KG != 0 && grp >= ktiles % KG) __syncthreads();
    }

    if constexpr (KG > 1) {
        // The groups' sums into LDS (their stages are free: every step ends
        // with a barrier), then group g adds up fragments g, g + KG, ... in
        // group order and finishes them.
        doublex4 *red = reinterpret_cast<doublex4 *>(lds);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) red[((grp * FM + i) * FN + j) * NT + t] = acc[i][j];
        __syncthreads();
#pragma unroll 1
        for (int q = grp; q < FM * FN; q += KG) {
            doublex4 sum = red[q * NT + t];
#pragma unroll
            for (int h = 1; h < KG; ++h) sum += red[(h * FM * FN + q) * NT + t];
            const int mb = m0 + wm * CF::WTM + (q / FN) * 16 + (lane >> 4);
            const int n = n0 + wn * CF::WTN + (q % FN) * 16 + (lane & 15);
            double cv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                cv[r] = (beta != 0.0 && mb + 4 * r < M && n < N) ? C[(long)(mb + 4 * r) * ldc + n] : 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (mb + 4 * r < M && n < N)
                    C[(long)(mb + 4 * r) * ldc + n] = (beta == 0.0) ? alpha * sum[r] : fma(alpha, sum[r], beta * cv[r]);
        }
        return;
    }

    // C values of one fragment row are loaded before any is stored (a load
    // cannot pass a possibly aliasing store: one latency per row, not per element).
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int mb = m0 + wm * CF::WTM + i * 16 + (lane >> 4);
        double cv[FN][4];
        if (beta != 0.0) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int n = n0 + wn * CF::WTN + j * 16 + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cv[j][r] = (interior || (mb + 4 * r < M && n < N)) ? C[(long)(mb + 4 * r) * ldc + n] : 0.0;
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * CF::WTN + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = mb + 4 * r;
                if (interior || (m < M && n < N))
                    C[(long)m * ldc + n] = (beta == 0.0) ? alpha * acc[i][j][r]
                                                         : fma(alpha, acc[i][j][r], beta * cv[j][r]);
            }
        }
    }
}

using D0 = DCfg<128, 128>;
using D1 = DCfg<64, 64>;
using D2 = DCfg<128, 64>;
using D3 = DCfg<64, 128>;
// Small grids (launch_small): K dealt to groups of one workgroup.
using D1K4 = DCfg<64, 64, 2, 4, 4>;
using D1S8 = DCfg<32, 32, 1, 8, 2>;
const char *kNames[] = {"f64_mfma_128x128x16", "f64_mfma_64x64x16", "f64_mfma_128x64x16", "f64_mfma_64x128x16"};
constexpr int kNum = 4;

template <class CF>
int launch_cfg(const Gemm<double> &g, hipStream_t s) {
    const int tiles_m = (g.M + CF::BM - 1) / CF::BM, tiles_n = (g.N + CF::BN - 1) / CF::BN;
    const long nblk = (long)tiles_m * tiles_n;
    if (nblk > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "dgemm: too many tiles (%ld)", nblk);
    int kc = g.K;
    const int splits = split_count(g.splits, nblk, g.K, 64, &kc, 2);
    double *ws = nullptr;
    if (splits > 1) {
        const int rc = stream_alloc((void **)&ws, (size_t)splits * g.M * g.N * sizeof(double), s);
        if (rc) return rc;
    }
    dim3 grid((unsigned)nblk, (unsigned)splits), block(CF::NT * CF::KG);
#define UGEMM_L(TA, TB) \
    hipLaunchKernelGGL((dgemm_mfma_kernel<CF, TA, TB>), grid, block, 0, s, g.M, g.N, g.K, g.alpha, g.A, \
                       g.lda, g.B, g.ldb, g.beta, g.C, g.ldc, tiles_m, tiles_n, kc, ws)
    timing_begin(s);
    if (!g.ta && !g.tb) UGEMM_L(false, false);
    else if (!g.ta && g.tb) UGEMM_L(false, true);
    else if (g.ta && !g.tb) UGEMM_L(true, false);
    else UGEMM_L(true, true);
    timing_end(s);
#undef UGEMM_L
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "dgemm launch");
    if (splits > 1) {
        if (!rc) rc = launch_splitk_reduce_f64(g.M, g.N, splits, g.alpha, ws, g.beta, g.C, g.ldc, s);
        const int rc2 = stream_free(ws, s);
        if (!rc) rc = rc2;
    }
    return rc;
}

// Variant 1 with the automatic split count: K dealt to groups of a workgroup
// where the grid leaves a CU one wave a SIMD (the reasons stand at the FP32
// kernel's launch_small; here 139 KB of LDS leave room for one workgroup of 8
// groups of 32x32 or of 4 groups of 64x64).  us a call, 64x64x1 / 64x64x4 / 32x32x8:
//   128x96x200 19.8 / 15.2 / 8.6;  512x512x512 29.8 / 25.5 / 12.1;  36x64x971 73 / 47 / 20;
//   1023x1000x1023 89 / 53 / 78;  58x16704x512 (261 of 64x64) 54 / 57 / 69.
int launch_small(const Gemm<double> &g, hipStream_t s) {
    const long cus = device_cu_count();
    const long t32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32), t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (g.splits != 0 || t64 > 4 * cus) return launch_cfg<D1>(g, s);
    Gemm<double> h = g;
    h.splits = 1;
    if (t32 <= cus && t32 * g.K <= cus * 2048) {
        if (g.K > 640) h.splits = (int)std::max(1L, std::min({cus / t32, g.K / 256L, 16L}));
        return launch_cfg<D1S8>(h, s);
    }
    return deal_k(t64, g.K, 38.0, 1, sizeof(*g.C) * g.M * g.N, &h.splits) ? (h.splits = 1, launch_cfg<D1K4>(h, s)) : launch_cfg<D1>(h, s);
}

}  // namespace

int dgemm_variant_count() { return kNum; }
const char *dgemm_variant_name(int v) { return (v >= 0 && v < kNum) ? kNames[v] : nullptr; }

int dgemm_pick_variant(const Gemm<double> &g) {
    const long cus = device_cu_count();
    const long t128 = (long)((g.M + 127) / 128) * ((g.N + 127) / 128);
    const long t64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
    const int v = t128 >= 2 * cus ? 0 : t64 <= 4 * cus ? 1 : g.M >= 4L * g.N ? 2 : g.N >= 4L * g.M ? 3 : 1;
    if (t128 <= cus) return v;
    // The fullest CU decides, as in fp32_pick_variant: 3573x5177x2321 NN on
    // 128x128 (five on a CU for 4.5 on average) 1827 us, on 128x64 1503;
    // 6240x1452x454 NT 227, on 64x64 172.
    static const TileCost cost[4] = {{128, 128, 100, 0}, {64, 64, 100, 0}, {128, 64, 97, 0}, {64, 128, 98, 0}};
    return cheapest_tile(cost, 4, 0, v, g.M, g.N);
}

int launch_dgemm(const Gemm<double> &g, int variant, hipStream_t s) {
    switch (variant) {
        case 0: return launch_cfg<D0>(g, s);
        case 1: return launch_small(g, s);
        case 2: return launch_cfg<D2>(g, s);
        case 3: return launch_cfg<D3>(g, s);
        default: return fail(UGEMM_ERR_ARG, "dgemm: no variant %d", variant);
    }
}

}  // namespace ugemm
