// The plain FP32 tile computation, shared by the single-GEMM kernel
// (sgemm_fp32.hip) and the grouped persistent kernel (grouped.hip).
//
// One workgroup computes one BM x BN tile of C:
//   * global -> registers -> LDS, two LDS stages: tile k+1 is fetched into
//     registers while tile k is multiplied from LDS, one barrier per BK step;
//   * LDS holds both operands K-major: As[k][m], Bs[k][n]; the transposed
//     layouts are turned around while writing LDS (no separate transpose pass);
//   * each thread owns a TM x TN register micro-tile built from 4-wide groups,
//     read from LDS with 128-bit loads; a wave is an 8 x 8 grid of threads, so a
//     k-step reads 128 contiguous bytes of As and of Bs per wave.
// Semantics follow the reference's row-major kernel gemm_rnn (sgemm_ocl2.h:17-90):
// C = alpha * acc + beta * C, C is not read when beta == 0 (sgemm_ocl2.h:86-88).
#pragma once

#include <type_traits>

#include "internal.h"
#include "conv_gather.h"
#include "kernel_common.h"

namespace ugemm {
namespace {

constexpr int LDS_PAD = 4;   // floats; keeps rows 16-byte aligned

// Empty register constraints on the accumulators.  They end a k-step: its
// FMAs must complete before the next step's code, which bounds live ranges.
// And they hold four columns j .. j + 3 of a row in one register quad rotated
// by one, column j + 3 first.  A v_fmac_f32 whose three operands lie in one
// register bank (number modulo 4) takes twice as long (measured with fixed
// registers: 63-75 against 123-141 TF/s for any other assignment).  Quads
// start at even registers, the fragments' as well as these, so a(i), b(j) and
// acc(i, j) could share a bank only if one quad started an odd distance from
// another in j: the rotation rules that out.  Left to the register allocator,
// 3-14% of the FMAs of a GEMM or convolution kernel had the conflict (counted in
// the assembly of each, 60 kernels; none has it now), and any change of the
// code around the loop moved that share.
template <int TM, int TN>
__device__ __forceinline__ void pin_step(float (&acc)[TM][TN]) {
    typedef float quad __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; j += 4) {
            quad q = {acc[i][j + 3], acc[i][j], acc[i][j + 1], acc[i][j + 2]};
            asm volatile("" : "+v"(q));
            acc[i][j + 3] = q[0];
            acc[i][j] = q[1];
            acc[i][j + 1] = q[2];
            acc[i][j + 2] = q[3];
        }
}

// MINB_: waves per SIMD the kernel is compiled for (register budget).
// KG_: groups of NT threads in a workgroup, each with its own LDS stages.
// Group g multiplies K tiles g, g + KG, ...; the groups' sums are added
// through LDS in group order.  For grids that leave CUs short of waves: one
// wave a SIMD hides no latency of its K steps.
template <int BM_, int BN_, int BK_, int TM_, int TN_, int MINB_ = 1, int KG_ = 1>
struct Fp32Cfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, TM = TM_, TN = TN_, MINB = MINB_;
    static constexpr int TX = BN / TN, TY = BM / TM;
    static constexpr int NT = TX * TY, KG = KG_, THREADS = NT * KG;
    static_assert(TM % 4 == 0 && TN % 4 == 0, "micro-tile built from 4-wide groups");
    static_assert(TX % 8 == 0 && TY % 8 == 0 && NT % 64 == 0, "waves are 8x8 thread grids");
    static constexpr int LDA = BM + LDS_PAD, LDB = BN + LDS_PAD;
    static constexpr int kStageFloats = 2 * BK * (LDA + LDB), kLdsFloats = KG * kStageFloats;   // two stages a group
    static_assert(KG == 1 || BM * BN <= kStageFloats, "the groups' sums fit their stages");
};

// One workgroup computes the C tile at (m0, n0) of g; shared by the plain and
// the grouped (persistent) kernels. lds must hold CF::kLdsFloats floats.
// CONV: opB is the implicit im2col matrix of cd (B and TB unused; ConvRegs).
// epi: bias and activation after alpha/beta (Epilogue, internal.h).
template <class CF, bool TA, bool TB, bool CONV = false>
__device__ __forceinline__ void fp32_tile(const int M, const int N, const int K, const float alpha,
                                          const float *__restrict__ A, const long lda,
                                          const float *__restrict__ B, const long ldb, const float beta,
                                          float *__restrict__ C, const long ldc, const int m0, const int n0,
                                          float *lds, const Epilogue &epi = Epilogue(),
                                          const ConvDesc &cd = ConvDesc()) {
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, TM = CF::TM, TN = CF::TN, NT = CF::NT;
    constexpr int LDA = CF::LDA, LDB = CF::LDB;
    constexpr int KG = CF::KG;
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);   // NT: whole waves
    float *As = lds + grp * CF::kStageFloats;   // [2][BK][LDA]
    float *Bs = As + 2 * BK * LDA;              // [2][BK][LDB]

    const int t = KG == 1 ? threadIdx.x : threadIdx.x % NT;
    const int lane = t & 63, w = t >> 6;
    constexpr int WX = CF::TX / 8;
    const int tx = (lane & 7) + 8 * (w % WX);
    const int ty = (lane >> 3) + 8 * (w / WX);

    // A tile: TA -> stored K x M (contiguous m); else M x K (contiguous k).
    using ARegs = TileRegs<float, TA ? BM : BK, TA ? BK : BM, NT>;
    using BRegs = TileRegs<float, TB ? BK : BN, TB ? BN : BK, NT>;
    ARegs ra;
    BRegs rb;

    const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
    const bool wide_a = (TA ? M : K) >= 4, wide_b = (TB ? K : N) >= 4;
    const int ktiles = (K + BK - 1) / BK;
    const int kfull = K / BK;   // tiles with no K tail

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
            ra.load_edge(a0, lda, t, TA ? mr : kr, TA ? kr : mr, wide_a);
            if constexpr (!CONV) rb.load_edge(b0, ldb, t, TB ? kr : nr, TB ? nr : kr, wide_b);
        }
        if constexpr (CONV) rc.load(cd, k0, K, t);
    };
    auto store_tile = [&](int kt, int buf, auto edge) {
        if constexpr (decltype(edge)::value) {
            const int mr = M - m0, nr = N - n0, kr = K - kt * BK;
            ra.mask(t, TA ? mr : kr, TA ? kr : mr, wide_a);
            if constexpr (!CONV) rb.mask(t, TB ? kr : nr, TB ? nr : kr, wide_b);
        }
        ra.template store<TA, LDA>(As + buf * BK * LDA, t);
        if constexpr (CONV) {
            rc.template store<LDB>(Bs + buf * BK * LDB, t);
        } else {
            rb.template store<!TB, LDB>(Bs + buf * BK * LDB, t);
        }
    };

    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = 0.0f;

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

    auto step = [&](int kt, int buf, bool more, auto edge) {   // edge: of the group's next K tile
        if (more) load_tile(kt + KG, edge);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front of the multiplications
        const float *as = As + buf * BK * LDA + ty * 4;
        const float *bs = Bs + buf * BK * LDB + tx * 4;
        // Register double-buffering of the k-step fragments: the LDS reads
        // of step k+1 are issued before the FMAs of step k. pin_step ends
        // each k-step: without it the compiler sinks all FMAs of the tile
        // below all of its LDS reads (4x the registers, spills).
        float a[2][TM], b[2][TN];
        auto read_frag = [&](int k, float *fa, float *fb) {
#pragma unroll
            for (int g = 0; g < TM / 4; ++g) {
                float4 x = *reinterpret_cast<const float4 *>(&as[k * LDA + g * CF::TY * 4]);
                fa[g * 4 + 0] = x.x; fa[g * 4 + 1] = x.y; fa[g * 4 + 2] = x.z; fa[g * 4 + 3] = x.w;
            }
#pragma unroll
            for (int g = 0; g < TN / 4; ++g) {
                float4 x = *reinterpret_cast<const float4 *>(&bs[k * LDB + g * CF::TX * 4]);
                fb[g * 4 + 0] = x.x; fb[g * 4 + 1] = x.y; fb[g * 4 + 2] = x.z; fb[g * 4 + 3] = x.w;
            }
        };
        read_frag(0, a[0], b[0]);
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            if (k + 1 < BK) read_frag(k + 1, a[(k + 1) & 1], b[(k + 1) & 1]);
            const float *fa = a[k & 1], *fb = b[k & 1];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) asm("v_fmac_f32 %0, %1, %2" : "+v"(acc[i][j]) : "v"(fa[i]), "v"(fb[j]));
            pin_step(acc);
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

    // Epilogue: C = alpha * acc (+ beta * C), then bias and activation, of
    // four columns n .. n + 3 of row m.
    const bool has_epi = epi.active();
    auto finish = [&](int m, int n, const f32x4u &q) {
        float *cp = C + (long)m * ldc + n;
        if (interior) {
            f32x4u o;
            if (beta == 0.0f) {
                o = alpha * q;
            } else {
                const f32x4u c = *reinterpret_cast<const f32x4u *>(cp);
                o = f32x4u{fmaf(alpha, q.x, beta * c.x), fmaf(alpha, q.y, beta * c.y), fmaf(alpha, q.z, beta * c.z),
                           fmaf(alpha, q.w, beta * c.w)};
            }
            if (has_epi) {
                o.x = apply_epilogue(epi, o.x, m, n);
                o.y = apply_epilogue(epi, o.y, m, n + 1);
                o.z = apply_epilogue(epi, o.z, m, n + 2);
                o.w = apply_epilogue(epi, o.w, m, n + 3);
            }
            *reinterpret_cast<f32x4u *>(cp) = o;
        } else if (m < M) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (n + j < N) {
                    float r = (beta == 0.0f) ? alpha * q[j] : fmaf(alpha, q[j], beta * cp[j]);
                    if (has_epi) r = apply_epilogue(epi, r, m, n + j);
                    cp[j] = r;
                }
            }
        }
    };
    constexpr int TG = TN / 4;
    if constexpr (KG == 1) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int g = 0; g < TG; ++g)
                finish(m0 + (i / 4) * CF::TY * 4 + ty * 4 + (i % 4), n0 + g * CF::TX * 4 + tx * 4,
                       f32x4u{acc[i][g * 4], acc[i][g * 4 + 1], acc[i][g * 4 + 2], acc[i][g * 4 + 3]});
    } else {
        // The groups' sums into LDS (their stages are free: every step ends
        // with a barrier), then group g adds up quads g, g + KG, ... of every
        // thread's micro-tile, in group order.
        typedef float quad __attribute__((ext_vector_type(4)));
        quad *red = reinterpret_cast<quad *>(lds);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int g = 0; g < TG; ++g)
                red[(grp * TM * TG + i * TG + g) * NT + t] =
                    quad{acc[i][g * 4], acc[i][g * 4 + 1], acc[i][g * 4 + 2], acc[i][g * 4 + 3]};
        __syncthreads();
#pragma unroll 1
        for (int q = grp; q < TM * TG; q += KG) {
            quad sum = red[q * NT + t];
#pragma unroll
            for (int h = 1; h < KG; ++h) sum += red[(h * TM * TG + q) * NT + t];
            const int i = q / TG, g = q % TG;
            finish(m0 + (i / 4) * CF::TY * 4 + ty * 4 + (i % 4), n0 + g * CF::TX * 4 + tx * 4,
                   f32x4u{sum.x, sum.y, sum.z, sum.w});
        }
    }
}

}  // namespace
}  // namespace ugemm
