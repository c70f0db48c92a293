// The FP32-MFMA tile computation (v_mfma_f32_16x16x4_f32), shared by the
// single-GEMM kernel (sgemm_mfma32.hip) and the grouped persistent kernel
// (grouped.hip).  FP32 operands as given, FP32 products, FP32 accumulation.
//
// A workgroup of WGM x WGN waves computes a BM x BN tile of C; each wave owns
// a (BM/WGM) x (BN/WGN) grid of 16x16 fragments.  Operand tiles of BK move
// global -> registers -> LDS, two LDS stages, one barrier per BK step.  Each
// operand keeps its global orientation in LDS, so every LDS store is a
// 16-byte vector store (no transposing writes):
//   k-contiguous operand (A when op(A) = A, B when op(B) = B^T): L[row][k],
//     row length BK + 4 floats; a lane reads its four k values as one
//     16-byte ds_read;
//   row-contiguous operand: L[k][row], row length rows + 4 floats; a lane
//     reads four single floats, 16 lanes over 64 contiguous bytes.
// The 16x16x4 MFMA takes from lane l the element (row l%16, k l/16).  Within
// a 16-deep k slab the lane's k group g = l/16 supplies k = 4g + q to the
// q-th MFMA (q = 0..3): both operands use this same permutation of k, so
// the sum over the slab is unchanged, and a lane's four k values are
// adjacent in memory for the k-contiguous layout.  The D fragment holds rows
// 4*(l/16) + r, column l%16.
// Semantics as sgemm_cpu (ugemm.h:287-411) with the BLAS beta == 0 rule
// (C is not read), as gemm_cpu.h:119-123.
#pragma once

#include <type_traits>

#include "internal.h"
#include "conv_gather.h"
#include "kernel_common.h"

namespace ugemm {
namespace {

typedef float m32_floatx4 __attribute__((ext_vector_type(4)));

// MINB_: waves per SIMD the kernel is compiled for (register budget).
// KG_: groups of WGM x WGN waves in a workgroup, each with its own LDS stages;
// group g multiplies K tiles g, g + KG, ... and the groups' sums are added
// through LDS in group order (small grids, as Fp32Cfg).
template <int BM_, int BN_, int BK_, int WGM_, int WGN_, int MINB_ = 1, int KG_ = 1>
struct M32Cfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WGN = WGN_, MINB = MINB_;
    static constexpr int NT = 64 * WGM * WGN, KG = KG_, THREADS = NT * KG;
    static constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 16, FN = WTN / 16;
    static_assert(BK % 16 == 0 && WTM % 16 == 0 && WTN % 16 == 0, "fragment-aligned tile");
    // LDS row length and stage size (floats) of an operand tile of ROWS rows.
    template <bool KC, int ROWS>
    static constexpr int ld() { return KC ? BK + 4 : ROWS + 4; }
    template <bool KC, int ROWS>
    static constexpr int stage() { return KC ? ROWS * (BK + 4) : BK * (ROWS + 4); }
    // LDS floats of the largest layout (both operands k-contiguous).
    static constexpr int kLdsFloats = KG * 2 * (BM + BN) * (BK + 4);
    // Of one layout (two stages of both operands a group).
    template <bool TA, bool TB>
    static constexpr int lds_floats() { return KG * 2 * (stage<!TA, BM>() + stage<TB, BN>()); }
};

template <class CF>
struct IsM32 : std::false_type {};
template <int BM, int BN, int BK, int WGM, int WGN, int MINB, int KG>
struct IsM32<M32Cfg<BM, BN, BK, WGM, WGN, MINB, KG>> : std::true_type {};

// The lane's four k values (k .. k+3) of fragment row `row`.
template <bool KC, int LD>
__device__ __forceinline__ m32_floatx4 m32_frag4(const float *L, int row, int k) {
    if constexpr (KC) {
        return *reinterpret_cast<const m32_floatx4 *>(L + row * LD + k);
    } else {
        return m32_floatx4{L[k * LD + row], L[(k + 1) * LD + row], L[(k + 2) * LD + row], L[(k + 3) * LD + row]};
    }
}

// C[m0:m0+BM, n0:n0+BN] = alpha * op(A) op(B) + beta * C, then the epilogue.
// A and B point at the operands' origins (k = 0).  lds: CF::kLdsFloats
// floats, 16-byte aligned.
// CONV: op(B) is the implicit im2col matrix of cd (B and TB unused; the
// gather of sgemm_gl1.h:166-190, ConvRegs); the B stage is [k][n].
template <class CF, bool TA, bool TB, bool CONV = false>
__device__ __forceinline__ void m32_tile(const int M, const int N, const int K, const float alpha,
                                         const float *__restrict__ A, const long lda, const float *__restrict__ B,
                                         const long ldb, const float beta, float *__restrict__ C, const long ldc,
                                         const int m0, const int n0, float *lds, const Epilogue &epi = Epilogue(),
                                         const ConvDesc &cd = ConvDesc()) {
    constexpr bool KCA = !TA, KCB = TB;
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, NT = CF::NT, FM = CF::FM, FN = CF::FN;
    constexpr int LDA = CF::template ld<KCA, BM>(), LDB = CF::template ld<KCB, BN>();
    constexpr int SA = CF::template stage<KCA, BM>(), SB = CF::template stage<KCB, BN>();
    constexpr int KG = CF::KG;
    static_assert(KG * 2 * (SA + SB) <= CF::kLdsFloats, "LDS budget");
    static_assert(KG == 1 || BM * BN <= 2 * (SA + SB), "the groups' sums fit their stages");
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    float *As = lds + grp * 2 * (SA + SB), *Bs = As + 2 * SA;
    const bool has_epi = epi.active();

    const int t = KG == 1 ? threadIdx.x : threadIdx.x % NT, lane = t & 63, w = t >> 6;
    const int wm = w / CF::WGN, wn = w % CF::WGN;

    using ARegs = TileRegs<float, KCA ? BK : BM, KCA ? BM : BK, NT>;
    using BRegs = TileRegs<float, KCB ? BK : BN, KCB ? BN : BK, NT>;
    ARegs ra;
    BRegs rb;
    const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
    const bool wide_a = (TA ? M : K) >= 4, wide_b = (TB ? K : N) >= 4;
    const int ktiles = (K + BK - 1) / BK, kfull = K / BK;

    // Implicit im2col operand (columns past N and taps outside the image read zeros).
    static_assert(!CONV || !TB, "implicit operand layout");
    using CRegs = typename ConvRegsOf<CONV, BK, BN, NT>::type;
    CRegs rc;
    if constexpr (CONV) rc.init(cd, n0 + t % BN, N);

    // EDGE tiles reach past M, N or K.
    auto load_tile = [&](int kt, auto edge) {
        const int k0 = kt * BK;
        const float *a0 = TA ? A + (long)k0 * lda + m0 : A + (long)m0 * lda + k0;
        const float *b0 = TB ? B + (long)n0 * ldb + k0 : B + (long)k0 * ldb + n0;
        if constexpr (!decltype(edge)::value) {
            ra.load(a0, lda, t);
            if constexpr (!CONV) rb.load(b0, ldb, t);
        } else {
            const int mr = M - m0, nr = N - n0, kr = K - k0;
            ra.load_edge(a0, lda, t, KCA ? kr : mr, KCA ? mr : kr, wide_a);
            if constexpr (!CONV) rb.load_edge(b0, ldb, t, KCB ? kr : nr, KCB ? nr : kr, wide_b);
        }
        if constexpr (CONV) rc.load(cd, k0, K, t);
    };
    auto store_tile = [&](int kt, int buf, auto edge) {
        if constexpr (decltype(edge)::value) {
            const int mr = M - m0, nr = N - n0, kr = K - kt * BK;
            ra.mask(t, KCA ? kr : mr, KCA ? mr : kr, wide_a);
            if constexpr (!CONV) rb.mask(t, KCB ? kr : nr, KCB ? nr : kr, wide_b);
        }
        ra.template store<true, LDA>(As + buf * SA, t);
        if constexpr (CONV) {
            rc.template store<LDB>(Bs + buf * SB, t);
        } else {
            rb.template store<true, LDB>(Bs + buf * SB, t);
        }
    };

    m32_floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = m32_floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // K tiles below nfast are loaded without bounds; the others (all of an
    // edge tile's, and a K remainder) as edges, in a loop of their own.
    const int nfast = (CONV ? m0 + BM <= M : interior) ? kfull : 0;
    if (grp < nfast) {
        load_tile(grp, std::false_type());
        store_tile(grp, 0, std::false_type());
    } else if (grp < ktiles) {
        load_tile(grp, std::true_type());
        store_tile(grp, 0, std::true_type());
    }
    __syncthreads();

    const int frow = lane & 15, g4 = (lane >> 4) * 4;
    auto step = [&](int kt, int buf, bool more, auto edge) {   // edge: of the group's next K tile
        if (more) load_tile(kt + KG, edge);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front of the multiplications
        const float *as = As + buf * SA, *bs = Bs + buf * SB;
#pragma unroll
        for (int s = 0; s < BK / 16; ++s) {
            m32_floatx4 fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[i] = m32_frag4<KCA, LDA>(as, wm * CF::WTM + i * 16 + frow, s * 16 + g4);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[j] = m32_frag4<KCB, LDB>(bs, wn * CF::WTN + j * 16 + frow, s * 16 + g4);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i][q], fb[j][q], acc[i][j], 0, 0, 0);
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
        m32_floatx4 *red = reinterpret_cast<m32_floatx4 *>(lds);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) red[((grp * FM + i) * FN + j) * NT + t] = acc[i][j];
        __syncthreads();
#pragma unroll 1
        for (int q = grp; q < FM * FN; q += KG) {
            m32_floatx4 sum = red[q * NT + t];
#pragma unroll
            for (int h = 1; h < KG; ++h) sum += red[(h * FM * FN + q) * NT + t];
            const int mb = m0 + wm * CF::WTM + (q / FN) * 16 + 4 * (lane >> 4);
            const int n = n0 + wn * CF::WTN + (q % FN) * 16 + (lane & 15);
            float cv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                cv[r] = (beta != 0.0f && mb + r < M && n < N) ? C[(long)(mb + r) * ldc + n] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (mb + r < M && n < N) {
                    float v = (beta == 0.0f) ? alpha * sum[r] : fmaf(alpha, sum[r], beta * cv[r]);
                    if (has_epi) v = apply_epilogue(epi, v, mb + r, n);
                    C[(long)(mb + r) * ldc + n] = v;
                }
        }
        return;
    }

    // C values of one fragment row are loaded before any is stored (a load
    // cannot pass a possibly aliasing store: one latency per row, not per element).
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int mb = m0 + wm * CF::WTM + i * 16 + 4 * (lane >> 4);
        float cv[FN][4];
        if (beta != 0.0f) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int n = n0 + wn * CF::WTN + j * 16 + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cv[j][r] = (interior || (mb + r < M && n < N)) ? C[(long)(mb + r) * ldc + n] : 0.0f;
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * CF::WTN + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = mb + r;
                if (interior || (m < M && n < N)) {
                    float v = (beta == 0.0f) ? alpha * acc[i][j][r] : fmaf(alpha, acc[i][j][r], beta * cv[j][r]);
                    if (has_epi) v = apply_epilogue(epi, v, m, n);
                    C[(long)m * ldc + n] = v;
                }
            }
        }
    }
}

}  // namespace
}  // namespace ugemm
