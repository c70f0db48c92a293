// Split SGEMM on gfx950 MFMA (v_mfma_f32_16x16x32_bf16 / _f16), FP32 accumulate.
//
// Splitting: every FP32 operand x is written as
//   x = h0 + h1 + h2 + r,  h0 = E(x), h1 = E(x - h0), h2 = E(x - h0 - h1)
// in a 16-bit element format E (round-to-nearest-even; the differences are
// exact in FP32).  NP planes are kept and the products
//   NP = 1 (BF16X1): h0*h0
//   NP = 2 (BF16X3): h0*h0 + h0*h1 + h1*h0                  |error| <~ 3*2^-16 |a||b|
//   NP = 3 (BF16X6): + h1*h1 + h0*h2 + h2*h0                |error| <~ 6*2^-24 |a||b|
// are issued as MFMAs into one FP32 accumulator, smallest terms first.
// Products of 16-bit values are exact in FP32, so the remaining error is the
// dropped terms plus FP32 accumulation.
//
// E = bf16 (8 significant bits) has FP32's exponent range and needs no
// scaling.  E = fp16 (11 significant bits: FP16X3, the NP = 2 products, error
// <~ 3*2^-22 |a||b|) has a narrow exponent range, so every row of op(A) and
// every column of op(B) is first scaled by a power of two 2^-e, e =
// exponent(max |x| of that row) - 15, bringing its largest magnitude into
// [2^14, 2^15) (exact: only the exponent changes); the epilogue multiplies
// C(m, n) by 2^(e_m + e_n) with ldexp, which is exact unless the true result
// itself over- or underflows.  Elements more than 2^28 below their row's
// maximum lose low-order bits to fp16 subnormals; their products are at most
// 2^-28 of the row's largest, so the effect on C is below 2^-40 |a||b|.
//
// Two kernels per call:
//  1. split_prep (HBM-bound): reads op(A) / op(B) once in any layout and
//     writes NP bf16 planes in "NT" form -- rows of A (m) and of B (n), k
//     contiguous -- zero-padded to whole tiles, so that the core needs no
//     bounds checks and no layout variants.  Transposed sources go through
//     an LDS tile so both the read and the write are coalesced.
//  2. split_nt_core (MFMA-bound): one workgroup per BM x BN tile of C, 4 waves
//     (2 x 2), each wave a (BM/2) x (BN/2) grid of 16x16 fragments whose
//     FP32 accumulators live in AGPRs; per K step of BK, all NP planes of the
//     A and B tiles are staged global -> registers -> LDS (two stages, the
//     next one in flight during the MFMAs), and every fragment read from LDS
//     serves every product that uses its plane.
// Fragment layout (16x16x32 bf16): lane l holds row l%16, k = 8*(l/16)..+7
// of A and the same k of column l%16 of B; D holds rows 4*(l/16)+i, column
// l%16.  A and B use the same k assignment, so any order of the hardware's
// internal sum pairs the right elements.
#include <string>
#include <type_traits>
#include <utility>

#include "internal.h"
#include "kernel_common.h"
#include "split_common.h"

namespace ugemm {
namespace {

// row_inf (scaled formats): the row's largest magnitude is infinite.
template <int NP, class FMT>
__device__ __forceinline__ void write_planes(typename FMT::E *dst, long plane_stride, const float (&x)[8],
                                             bool row_inf = false) {
    typename FMT::V8 w[NP];
    split8<NP, FMT>(x, __any(split_special(FMT(), x, row_inf)), w);
#pragma unroll
    for (int p = 0; p < NP; ++p) *reinterpret_cast<typename FMT::V8 *>(dst + p * plane_stride) = w[p];
}

// Plane layout written by the preparation kernels ("k-tile blocked"): plane
// p of an operand with rows_pad rows and k_pad (multiple of 32) columns holds
// element (r, k) at
//   p * plane_stride + ((k / 32) * rows_pad + r) * 32 + (chunk ^ sw(r)) * 8 + k % 8,
// chunk = (k % 32) / 8, sw(r) = (r >> 1) & 3.  One K tile of BM rows is thus a
// contiguous BM * 64-byte block whose bytes are already in the (bank-conflict
// free, see swz_chunk) order of the LDS stage: the core copies it verbatim.
__device__ __forceinline__ long blocked_offset(int r, int k, int rows_pad) {
    return ((long)(k >> 5) * rows_pad + r) * 32 + ((((k >> 3) & 3) ^ ((r >> 1) & 3)) << 3);
}

// Source element (r, k) of the operand: X[r*ld + k] (k-contiguous) or
// X[k*ld + r] (row-contiguous); zeros outside rows x K.  FMT::SCALED: row r is
// multiplied by 2^-row_exp(amax[r]) before splitting.

// k-contiguous source, 2-D blocks: block (bx, by) covers rows [64 bx, +64)
// and k [128 by, +128) (four 32-wide k tiles).  Chunk f = t + 256 i of a
// thread is row f / 16, k-chunk f % 16: each load instruction of a wave reads
// four 512-byte row segments, and each store writes four 256-byte runs of
// the blocked layout (the rows of one k tile are contiguous there) -- where
// a row-major walk stored sixteen 64-byte pieces per instruction.  All four
// chunks are loaded before any is split.
template <int NP, class FMT>
__device__ __forceinline__ void prep_kcont_tile(const float *__restrict__ X, long ld, int rows, int K, typename FMT::E *__restrict__ out, long plane_stride, int rows_pad,
                                                int k_pad, const unsigned *__restrict__ amax, int r0, int k0) {
    const int t = threadIdx.x;
    // Scaled formats: the row maxima are loaded first, so that their latency
    // overlaps the operand loads instead of following them.
    unsigned am[4] = {0u, 0u, 0u, 0u};
    if constexpr (FMT::SCALED) {
#pragma unroll
        for (int i = 0; i < 4; ++i) am[i] = amax[r0 + ((t + 256 * i) >> 4)];
    }
    float x[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = t + 256 * i, r = r0 + (f >> 4), k = k0 + (f & 15) * 8;
        const float *p = X + (long)r * ld + k;
        if (r < rows && k + 8 <= K) {
            const f32x4u a = *reinterpret_cast<const f32x4u *>(p);
            const f32x4u b = *reinterpret_cast<const f32x4u *>(p + 4);
            x[i][0] = a.x; x[i][1] = a.y; x[i][2] = a.z; x[i][3] = a.w;
            x[i][4] = b.x; x[i][5] = b.y; x[i][6] = b.z; x[i][7] = b.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[i][j] = (r < rows && k + j < K) ? p[j] : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = t + 256 * i, r = r0 + (f >> 4), k = k0 + (f & 15) * 8;
        if (k >= k_pad) continue;
        if constexpr (FMT::SCALED) {
            const int e = -row_exp(am[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[i][j] = ldexpf(x[i][j], e);
        }
        write_planes<NP, FMT>(out + blocked_offset(r, k, rows_pad), plane_stride, x[i], row_is_inf(am[i]));
    }
}

// FP16X3, k-contiguous source with k_pad <= 8192: the row maximum and the
// split in one pass.  Block b reads rows r0 = 2b and r0 + 1 once into
// registers, reduces each row's largest magnitude (amax[r], as the separate
// row-maximum pass computes it: NaN ignored, 0 for padding rows), then
// scales by 2^-row_exp and writes the planes -- the operand is read once
// instead of twice.  Two rows per block, so that their 64-byte segments of
// a K tile -- adjacent in the blocked layout -- leave as one 128-byte line
// (one row per block: 0.172 against 0.138 ms at 8192^3 for the launch below
// that also scans B): thread t takes 8-k chunk t % 4 of row r0 + (t / 4) % 2
// in K tile t / 8 of each 32-tile pass (at most 8 passes, k_pad <= 8192).
// Each row's maximum is reduced over the lanes that hold it (shuffles that
// keep bit 2 of the lane fixed), then over the waves.
// lanes (16 .. 256, a power of two): threads to a pair of rows.  Rows of fewer
// than 32 K tiles leave the rest of the block to further pairs (row_lanes;
// 30564x448x49: 85 us a call before, 38 now).
inline int row_lanes(int k_pad) {   // 8 a K tile; k_pad is a multiple of 64
    int lanes = 16;
    while (lanes < 256 && lanes * 4 < k_pad) lanes *= 2;
    return lanes;
}

template <int NP, class FMT>
__device__ __forceinline__ void prep_kcont_rowscaled_pair(const float *__restrict__ X, long ld, int rows, int K,
                                                          typename FMT::E *__restrict__ out,
                                                          long plane_stride, int rows_pad, int k_pad,
                                                          unsigned *__restrict__ amax, int r0,
                                                          int lanes = 256) {
    static_assert(FMT::SCALED, "row scales");
    constexpr int PASSES = 8;   // 8 passes x 32 K tiles x 32 = 8192
    const int t = threadIdx.x & (lanes - 1), group = threadIdx.x / lanes;
    const int ktl = t >> 3, rr = (t >> 2) & 1, cc = t & 3, r = r0 + 2 * group + rr;
    const int ktiles = k_pad / 32;
    float x[PASSES][8];
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int kt = i * 32 + ktl, k = kt * 32 + cc * 8;
        const float *p = X + (long)r * ld + k;
        if (kt < ktiles && r < rows && k + 8 <= K) {
            const f32x4u a = *reinterpret_cast<const f32x4u *>(p);
            const f32x4u c = *reinterpret_cast<const f32x4u *>(p + 4);
            x[i][0] = a.x; x[i][1] = a.y; x[i][2] = a.z; x[i][3] = a.w;
            x[i][4] = c.x; x[i][5] = c.y; x[i][6] = c.z; x[i][7] = c.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[i][j] = (kt < ktiles && r < rows && k + j < K) ? p[j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(x[i][j]));
    }
    m = fmaxf(m, __shfl_xor(m, 1));
    m = fmaxf(m, __shfl_xor(m, 2));
    m = fmaxf(m, __shfl_xor(m, 8));
    if (lanes > 16) m = fmaxf(m, __shfl_xor(m, 16));
    if (lanes > 32) m = fmaxf(m, __shfl_xor(m, 32));
    if (lanes > 64) {   // uniform: 2 or 4 waves a group
        __shared__ float wmax[4][2];
        if ((t & 63) < 8 && (t & 3) == 0) wmax[threadIdx.x >> 6][rr] = m;
        __syncthreads();
        const int w0 = group * (lanes >> 6);
        m = fmaxf(wmax[w0][rr], wmax[w0 + 1][rr]);
        if (lanes == 256) m = fmaxf(m, fmaxf(wmax[2][rr], wmax[3][rr]));
    }
    const unsigned bits = m > 0.0f ? __float_as_uint(m) : 0u;
    if (t < 8 && (t & 3) == 0) amax[r] = bits;
    const int e = -row_exp(bits);
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int kt = i * 32 + ktl;
        if (kt >= ktiles) break;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[i][j] = ldexpf(x[i][j], e);
        write_planes<NP, FMT>(out + blocked_offset(r, kt * 32 + cc * 8, rows_pad), plane_stride, x[i],
                              row_is_inf(bits));
    }
}

// Partial row maxima of a row-contiguous operand, at most (FP16X3).
constexpr int kAmaxParts = 16;

// Row-contiguous source (X[k*ld + r]): the 64 x 64 tile (rows r0.., k k0..)
// transposed through LDS (tile[64][65], 256 threads).
template <int NP, class FMT>
__device__ __forceinline__ void prep_rcont_tile(const float *__restrict__ X, long ld, int rows, int K, typename FMT::E *__restrict__ out, long plane_stride, int rows_pad,
                                                int k_pad, const unsigned *__restrict__ amax, int r0, int k0,
                                                float (*tile)[65], const unsigned *__restrict__ parts = nullptr,
                                                int nparts = 0) {
    const int t = threadIdx.x;
    // Scaled formats: this thread's two row maxima, loaded before the tile; or
    // (parts) its share of one row's, put together behind the tile's barrier.
    unsigned am[2] = {0u, 0u}, pm[kAmaxParts / 4];
    __shared__ unsigned pmax[FMT::SCALED ? 4 : 1][FMT::SCALED ? 64 : 1];
    if constexpr (FMT::SCALED) {
        if (nparts) {
            const int r = min(r0 + (t & 63), rows - 1);   // repeats change no maximum; past the rows it is not used
#pragma unroll
            for (int i = 0; i < kAmaxParts / 4; ++i)
                pm[i] = parts[(long)min((t >> 6) + 4 * i, nparts - 1) * rows_pad + r];
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = r0 + (t + i * 256) / 8;
                am[i] = r < rows_pad ? amax[r] : 0u;
            }
        }
    }
    // Read: 64 k-lines of 64 r each, as 16 float4 per line (coalesced along r).
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = t + i * 256;
        const int kk = f / 16, rr = (f % 16) * 4;
        const int k = k0 + kk, r = r0 + rr;
        const float *p = X + (long)k * ld + r;
        float v[4];
        if (k < K && r + 4 <= rows) {
            const f32x4u a = *reinterpret_cast<const f32x4u *>(p);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (k < K && r + j < rows) ? p[j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[kk][rr + j] = v[j];
    }
    if constexpr (FMT::SCALED) {
        if (nparts) pmax[t >> 6][t & 63] = max(max(pm[0], pm[1]), max(pm[2], pm[3]));
    }
    __syncthreads();
    if constexpr (FMT::SCALED) {
        if (nparts) {
            auto row_max = [&](int r) { return max(max(pmax[0][r], pmax[1][r]), max(pmax[2][r], pmax[3][r])); };
#pragma unroll
            for (int i = 0; i < 2; ++i) am[i] = row_max((t + i * 256) / 8);
            if (k0 == 0 && t < 64 && r0 + t < rows_pad) const_cast<unsigned *>(amax)[r0 + t] = row_max(t);
        }
    }
    // Write: 64 rows of 8 chunks of 8 k.
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int f = t + i * 256;
        const int rr = f / 8, kk = (f % 8) * 8;
        const int r = r0 + rr, k = k0 + kk;
        if (r >= rows_pad || k >= k_pad) continue;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = tile[kk + j][rr];
        if constexpr (FMT::SCALED) {
            const int e = -row_exp(am[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = ldexpf(x[j], e);
        }
        write_planes<NP, FMT>(out + blocked_offset(r, k, rows_pad), plane_stride, x, row_is_inf(am[i]));
    }
}

// block_job[b]: the job of preparation block b (one load, where a search of
// the job table took ~10 dependent loads per block).  A block prepares
// kPrepSpan consecutive k tiles of one 64-row stripe (fewer job lookups and
// block starts per byte): 64-row x 128-k tiles of a k-contiguous job
// (prep_kcont_tile: four 512-byte row segments per load instruction,
// 256-byte runs per store), 64 x 64 transposing tiles of a row-contiguous
// one; nbx blocks along the rows.
template <int NP, class FMT>
__global__ __launch_bounds__(256) void grouped_split_prep(const PrepJob *__restrict__ jobs,
                                                          const int *__restrict__ block_job) {
    __shared__ float tile[64][65];
    const PrepJob j = jobs[block_job[blockIdx.x]];
    const int lb = (int)blockIdx.x - j.block0;
    typename FMT::E *out = static_cast<typename FMT::E *>(j.out);
    if constexpr (FMT::SCALED) {
        if (j.kcont == kPrepRowScaled) {
            // The maxima buffer is the plan's own device memory, written here.
            prep_kcont_rowscaled_pair<NP, FMT>(j.X, j.ld, j.rows, j.K, out, j.plane_stride, j.rows_pad,
                                               j.k_pad, const_cast<unsigned *>(j.amax), lb * 2);
            return;
        }
    }
    const int r0 = (lb % j.nbx) * 64, kb = (lb / j.nbx) * kPrepSpan;
    if (j.kcont) {
        for (int s = 0; s < kPrepSpan && (kb + s) * 128 < j.k_pad; ++s)
            prep_kcont_tile<NP, FMT>(j.X, j.ld, j.rows, j.K, out, j.plane_stride, j.rows_pad, j.k_pad,
                                     j.amax, r0, (kb + s) * 128);
    } else {
        for (int s = 0; s < kPrepSpan && (kb + s) * 64 < j.k_pad; ++s) {
            if (s > 0) __syncthreads();   // the previous tile's reads of the LDS tile are done
            prep_rcont_tile<NP, FMT>(j.X, j.ld, j.rows, j.K, out, j.plane_stride, j.rows_pad, j.k_pad,
                                     j.amax, r0, (kb + s) * 64, tile);
        }
    }
}

// Both operands of one GEMM in one launch (scaled formats: their maxima known):
// blocks [0, b.block0) prepare a, the rest b, one tile each (64-row x 128-k
// tiles of a k-contiguous operand, 64 x 64 transposing tiles of a
// row-contiguous one; nbx blocks along the rows).  One launch instead of
// two saves a launch and lets b's tiles start while a's last ones drain
// (2048^3 BF16x3: 263 against 256 TF/s per call).
template <int NP, class FMT>
__global__ __launch_bounds__(256) void split_prep_pair(PrepJob a, PrepJob b) {
    __shared__ float tile[64][65];
    const bool second = (int)blockIdx.x >= b.block0;
    const PrepJob &j = second ? b : a;
    const int lb = (int)blockIdx.x - j.block0;
    typename FMT::E *out = static_cast<typename FMT::E *>(j.out);
    const int r0 = (lb % j.nbx) * 64;
    if (j.kcont)
        prep_kcont_tile<NP, FMT>(j.X, j.ld, j.rows, j.K, out, j.plane_stride, j.rows_pad, j.k_pad,
                                 j.amax, r0, (lb / j.nbx) * 128);
    else
        prep_rcont_tile<NP, FMT>(j.X, j.ld, j.rows, j.K, out, j.plane_stride, j.rows_pad, j.k_pad,
                                 j.amax, r0, (lb / j.nbx) * 64, tile, j.parts, j.nparts);
}

// Largest magnitude of every plane row (row r of op(A), column r of op(B))
// as IEEE bits, combined with atomicMax on the bit pattern (non-negative
// floats order like their bit patterns).  amax must be zeroed first.
__global__ void fill_zero_u32(unsigned *__restrict__ p, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0u;
}

// k-contiguous source: block b covers row b / kchunks, k in [2048 * (b % kchunks), +2048).
// One chunk a row: stored, not combined, and the block may lie past the rows (0).
__device__ __forceinline__ void row_amax_kcont_block(const float *__restrict__ X, long ld, int rows, int K, long kchunks, unsigned *__restrict__ amax, long b) {
    const int r = (int)(b / kchunks);
    const int k = (int)(b % kchunks) * 2048 + threadIdx.x * 8;
    const float *p = X + (long)r * ld + k;
    float m = 0.0f;
    if (r < rows && k + 8 <= K) {
        const f32x4u a = *reinterpret_cast<const f32x4u *>(p);
        const f32x4u c = *reinterpret_cast<const f32x4u *>(p + 4);
        m = fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                  fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w))));
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (r < rows && k + j < K) m = fmaxf(m, fabsf(p[j]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    __shared__ float wmax[4];
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
        if (kchunks == 1) {
            amax[r] = m > 0.0f ? __float_as_uint(m) : 0u;
        } else if (r < rows && m > 0.0f) {
            atomicMax(&amax[r], __float_as_uint(m));
        }
    }
}

// Row-contiguous source (X[k*ld + r]): block b covers columns r in
// [4 CG (b % cblocks), +4 CG) and k in [S * (b / cblocks), +S), S =
// kAmaxRcontSpan, cblocks = ceil(rows / (4 CG)): consecutive blocks read
// neighbouring row segments (blocks that shared columns and differed only in
// k read addresses a power-of-two multiple of the row pitch apart, which crowd
// the same HBM channels).  CG = 64: 1 KB segments; CG = 16, four times the
// blocks, for operands that would leave CUs idle.  PARTS: row b / cblocks of
// the partial maxima (rows_pad long) instead of combined ones.
template <int CG, bool PARTS = false>
__device__ __forceinline__ void row_amax_rcont_block(const float *__restrict__ X, long ld, int rows, int K,
                                                     unsigned *__restrict__ amax, long b, long rows_pad = 0) {
    constexpr int COLS = 4 * CG, KP = 256 / CG, SPAN = kAmaxRcontSpan, PER = SPAN / KP, BATCH = PER < 16 ? PER : 16;
    const long cblocks = (rows + COLS - 1) / COLS;
    const int c0 = (int)(b % cblocks) * COLS, k0 = (int)(b / cblocks) * SPAN;
    const int cg = threadIdx.x % CG, kp = threadIdx.x / CG;
    const int c = c0 + cg * 4;
    float m[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (c + 4 <= rows && k0 + SPAN <= K) {
        // Whole block: PER independent 16-byte loads per thread, issued 16 at
        // a time into registers before any is used (the compiler otherwise
        // waits after every second load, which leaves HBM idle).
        const float *p = X + (long)(k0 + kp) * ld + c;
        for (int kb = 0; kb < PER; kb += BATCH) {
            f32x4u v[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) v[i] = *reinterpret_cast<const f32x4u *>(p + (long)(kb + i) * KP * ld);
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                m[0] = fmaxf(m[0], fabsf(v[i].x)); m[1] = fmaxf(m[1], fabsf(v[i].y));
                m[2] = fmaxf(m[2], fabsf(v[i].z)); m[3] = fmaxf(m[3], fabsf(v[i].w));
            }
        }
    } else {
        for (int kk = kp; kk < SPAN && k0 + kk < K; kk += KP) {
            const float *p = X + (long)(k0 + kk) * ld + c;
            if (c + 4 <= rows) {
                const f32x4u a = *reinterpret_cast<const f32x4u *>(p);
                m[0] = fmaxf(m[0], fabsf(a.x)); m[1] = fmaxf(m[1], fabsf(a.y));
                m[2] = fmaxf(m[2], fabsf(a.z)); m[3] = fmaxf(m[3], fabsf(a.w));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c + j < rows) m[j] = fmaxf(m[j], fabsf(p[j]));
            }
        }
    }
    __shared__ float sm[KP][COLS];
#pragma unroll
    for (int j = 0; j < 4; ++j) sm[kp][cg * 4 + j] = m[j];
    __syncthreads();
    const int t = threadIdx.x, col = c0 + t;
    if (t >= COLS || col >= rows) return;
    float v = sm[0][t];
#pragma unroll
    for (int i = 1; i < KP; ++i) v = fmaxf(v, sm[i][t]);
    if constexpr (PARTS) amax[(b / cblocks) * rows_pad + col] = v > 0.0f ? __float_as_uint(v) : 0u;
    else if (v > 0.0f) atomicMax(&amax[col], __float_as_uint(v));
}

// Before the planes of one FP16X3 GEMM, in one launch for both operands, so
// that their passes over HBM overlap: `none`, or whole rows of a k-contiguous
// operand to planes and maxima (prep_kcont_rowscaled_pair), or only its row
// maxima, or those of a row-contiguous operand (columns by 256 or 64, combined
// or in parts).
enum ScaleKind { SCALE_NONE, SCALE_SPLIT_ROWS, SCALE_KCONT, SCALE_RCONT, SCALE_RCONT_NARROW, SCALE_PARTS,
                 SCALE_PARTS_NARROW };
struct ScaleJob {
    const float *X;
    long ld, plane_stride, chunks;   // chunks: of 2048 a row; SCALE_SPLIT_ROWS: lanes
    void *out;
    unsigned *amax, *parts;
    int kind, rows, rows_pad, k_pad, blocks;
};
template <int NP, class FMT>
__global__ __launch_bounds__(256) void split_scales(ScaleJob a, ScaleJob b, int K) {
    const bool second = (int)blockIdx.x >= a.blocks;
    const ScaleJob &j = second ? b : a;
    const int lb = (int)blockIdx.x - (second ? a.blocks : 0);
    switch (j.kind) {
        case SCALE_SPLIT_ROWS:
            prep_kcont_rowscaled_pair<NP, FMT>(j.X, j.ld, j.rows, K, static_cast<typename FMT::E *>(j.out),
                                               j.plane_stride, j.rows_pad, j.k_pad, j.amax,
                                               lb * (int)(512 / j.chunks), (int)j.chunks);
            break;
        case SCALE_KCONT: row_amax_kcont_block(j.X, j.ld, j.rows, K, j.chunks, j.amax, lb); break;
        case SCALE_RCONT: row_amax_rcont_block<64>(j.X, j.ld, j.rows, K, j.amax, lb); break;
        case SCALE_RCONT_NARROW: row_amax_rcont_block<16>(j.X, j.ld, j.rows, K, j.amax, lb); break;
        case SCALE_PARTS: row_amax_rcont_block<64, true>(j.X, j.ld, j.rows, K, j.parts, lb, j.rows_pad); break;
        case SCALE_PARTS_NARROW: row_amax_rcont_block<16, true>(j.X, j.ld, j.rows, K, j.parts, lb, j.rows_pad); break;
        default: break;
    }
}

// Row maxima of the operands of a grouped FP16X3 plan: job j (PrepJob with
// out = its maxima, nbx = K chunks per row (k-contiguous: 2048 wide) or per
// 256-column block (row-contiguous: kAmaxRcontSpan deep)), blocks as in the kernels above.
__global__ __launch_bounds__(256) void grouped_row_amax(const PrepJob *__restrict__ jobs,
                                                        const int *__restrict__ block_job) {
    const PrepJob j = jobs[block_job[blockIdx.x]];
    const long lb = (long)blockIdx.x - j.block0;
    unsigned *amax = static_cast<unsigned *>(j.out);
    if (j.kcont) row_amax_kcont_block(j.X, j.ld, j.rows, j.K, j.nbx, amax, lb);
    else row_amax_rcont_block<64>(j.X, j.ld, j.rows, j.K, amax, lb);
}

// Implicit im2col operand of a convolution (ConvDesc): element (n, k) of the
// N x K operand (opB transposed) is in[c][ho*stride - pad + i][wo*stride - pad + j]
// for n = ho*wcol + wo and k = (c, i, j) = c*kk*kk + i*kk + j, zero outside the
// image and beyond N x K; ktab[k] = {c*H*W + i*W + j, (i << 16) | j}.  The
// gather follows sgemm_gl1.h:166-190 (see oracle_im2col).
__device__ __forceinline__ float im2col_at(const ConvDesc &cd, int n, int k, int N, int K) {
    if (n >= N || k >= K) return 0.0f;
    const int ho = n / cd.wcol, wo = n - ho * cd.wcol;
    const int h0 = ho * cd.stride - cd.pad, w0 = wo * cd.stride - cd.pad;
    const int2 e = cd.ktab[k];
    const int hi = h0 + (e.y >> 16), wi = w0 + (e.y & 0xffff);
    return ((unsigned)hi < (unsigned)cd.H && (unsigned)wi < (unsigned)cd.W) ? cd.in[(long)h0 * cd.W + w0 + e.x] : 0.0f;
}

// Planes of the im2col operand, gathered straight from the image (no im2col
// matrix in HBM): one thread per 8 k of one pixel n.
template <int NP, class FMT>
__global__ __launch_bounds__(256) void split_prep_im2col(ConvDesc cd, int N, int K, typename FMT::E *__restrict__ out,
                                                         long plane_stride, int rows_pad, int k_pad,
                                                         const unsigned *__restrict__ amax) {
    const long chunks_per_row = k_pad / 8;
    const long total = (long)rows_pad * chunks_per_row;
    for (long f = (long)blockIdx.x * blockDim.x + threadIdx.x; f < total; f += (long)gridDim.x * blockDim.x) {
        const int r = (int)(f / chunks_per_row);
        const int k = (int)(f - (long)r * chunks_per_row) * 8;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = im2col_at(cd, r, k + j, N, K);
        bool inf = false;
        if constexpr (FMT::SCALED) {
            const int e = -row_exp(amax[r]);
            inf = row_is_inf(amax[r]);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = ldexpf(x[j], e);
        }
        write_planes<NP, FMT>(out + blocked_offset(r, k, rows_pad), plane_stride, x, inf);
    }
}

// Largest magnitude of every pixel column of the im2col operand (scaled
// formats): thread n of block (bx, by) scans k in [by*kspan, +kspan).
__global__ __launch_bounds__(256) void row_amax_im2col(ConvDesc cd, int N, int K, int kspan,
                                                       unsigned *__restrict__ amax) {
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    const int k0 = blockIdx.y * kspan, k1 = min(K, k0 + kspan);
    float m = 0.0f;
    for (int k = k0; k < k1; ++k) m = fmaxf(m, fabsf(im2col_at(cd, n, k, N, K)));
    if (m > 0.0f) atomicMax(&amax[n], __float_as_uint(m));
}

// ---------------------------------------------------------------------------
// MFMA core over prepared planes.

// 16-byte chunk swizzle inside a plane row of CPR chunks: chunk c of row r is
// stored at c ^ sw(r), sw(r) = (r >> 1) & 3 (CPR 4) or r & 7 (CPR 8).
// Measured with SQ_LDS_BANK_CONFLICT on gfx950: fragment reads (16 lanes =
// 16 consecutive rows, one chunk each) are conflict-free with these.
template <int CPR>
__device__ __forceinline__ int swz_chunk(int row, int c) {
    if constexpr (CPR == 8) return c ^ (row & 7);
    else return c ^ ((row >> 1) & 3);
}

// First product (in Products order) that uses plane p of A / of B: the
// phased core reads a plane's fragments from LDS right before that product.
template <int NP>
constexpr bool first_use_a(int q) {
    for (int r = 0; r < q; ++r)
        if (Products<NP>::a[r] == Products<NP>::a[q]) return false;
    return true;
}
template <int NP>
constexpr bool first_use_b(int q) {
    for (int r = 0; r < q; ++r)
        if (Products<NP>::b[r] == Products<NP>::b[q]) return false;
    return true;
}

// WGM x WGN waves per workgroup.  PHASED: fragments of each plane are read
// just before the first product that needs them, behind a scheduling
// barrier, so that at most three planes' fragments are live (2 waves per
// SIMD fit in 256 registers); the other wave on the SIMD covers the LDS
// latency.  Otherwise all fragments of a K step are read first.
//
// ILV (phased variants with two LDS stages): stage kt+1 waits in registers
// during step kt.  Its LDS stores, and the global loads of stage kt+2 into
// the same registers, are interleaved with the MFMAs of the step's last
// product instead of running between the MFMAs and the barrier: the loads
// get a full step of latency and no wave stalls on a burst of stores in
// front of the barrier.  It needs the registers of 2 waves per SIMD.
// STREAM (required by ILV): each A fragment is read two MFMA groups (of FN
// MFMAs) ahead of its use, and the next product's B fragments during the
// current product's last groups, in an order that scheduling barriers fix.
// (Left to itself the compiler issued a product's reads in one burst and
// then waited on them.)  Every variant issues the same MFMAs per accumulator
// in the same order: results are bitwise identical across them.
// EARLY (with STREAM, for NP >= 2, whose last product reuses planes held in
// registers): the block barrier moves from the end of a K tile to the start
// of its last product.  The stage copy is dealt over the products before the
// barrier, so after it the last product's MFMAs cover the reads of the next
// K tile's first fragments (from the other buffer) instead of the tile
// starting on a burst of reads.
template <int BM_, int BN_, int BK_, int NP_, class FMT_ = FmtBf16, int WGM_ = 2, int WGN_ = 2, bool PHASED_ = false,
          bool ILV_ = false, bool STREAM_ = false, bool EARLY_ = false>
struct CoreCfg {
    using FMT = FMT_;
    static constexpr int BM = BM_, BN = BN_, BK = BK_, NP = NP_;
    static constexpr bool PHASED = PHASED_, ILV = ILV_, STREAM = STREAM_, EARLY = EARLY_;
    static constexpr int WGM = WGM_, WGN = WGN_, NT = 64 * WGM_ * WGN_;
    static constexpr int WTM = BM / WGM, WTN = BN / WGN;
    static constexpr int FM = WTM / 16, FN = WTN / 16;
    static constexpr int KSTEPS = BK / 32, CPR = BK / 8;
    static constexpr int A_PLANE = BM * BK, B_PLANE = BN * BK;           // bf16 elements
    static constexpr int STAGE = NP * (A_PLANE + B_PLANE);
    static constexpr int STAGES = (2 * STAGE * 2 <= 160 * 1024) ? 2 : 1;
    static constexpr int LDS_BYTES = STAGES * STAGE * 2;
    static constexpr int CHUNKS = NP * (BM + BN) * CPR;                 // 16-byte chunks per stage
    // 8-wave variants can also split a k-contiguous FP32 operand while
    // staging it (no preparation pass for that operand); 16 waves have no
    // registers to spare for it.
    static constexpr bool FUSABLE = 64 * WGM_ * WGN_ == 512;
    static constexpr int PER_T = CHUNKS / NT;
    static_assert(CHUNKS % NT == 0, "stage must split evenly over the threads");
    static_assert(WTM % 16 == 0 && WTN % 16 == 0 && BK % 32 == 0, "tile shape");
    static_assert(!ILV || (PHASED && STAGES == 2 && KSTEPS == 1), "interleaved staging needs phased reads, two stages");
    static_assert(ILV == STREAM && (!STREAM || FM >= 4), "the interleaved staging runs with streamed reads");
    static_assert(!EARLY || (STREAM && NP >= 2 && FN + 2 <= FM), "early reads: streamed, last product resident");
};

enum { FUSE_NONE = 0, FUSE_KCONT = 1, FUSE_RCONT = 2 };

// amax_a / amax_b: per-row largest magnitudes of the scaled formats
// (FMT::SCALED), unused otherwise.
// FA / FB (FUSE_*): where the core takes that operand's stage from.
//   FUSE_NONE:  prepared planes, copied verbatim.
//   FUSE_KCONT: split while staging from the k-contiguous FP32 source
//     X[r*ld + k].  Thread t handles the chunks f = t + NT*i of the stage
//     (row r = f / 4, stored chunk f % 4, which holds k-chunk (f % 4) ^ sw(r)).
//   FUSE_RCONT: split while staging from the row-contiguous FP32 source
//     X[k*ld + r], transposed in registers: thread t loads 8 k-lines of the
//     RPT adjacent rows rp*RPT .. rp*RPT + RPT - 1 (RPT = rows*4/NT, 1 or 2;
//     rp = t % (rows/RPT), k-chunk t / (rows/RPT)), coalesced along r, and
//     splits one 8-k chunk per row.
// Either way each split chunk lands where the plane copy would have put it
// (zeros beyond M, N, K).
// GR (grouped plans): block b computes tile gtiles[b] of problem
// gprobs[gtiles[b].problem], whose planes, sizes, alpha, beta and C (and,
// with FB, B's FP32 source) replace the corresponding arguments (no split K,
// no epilogue, A always from planes).
template <class CF, int FA, int FB, bool GR = false>
__global__ __launch_bounds__(CF::NT) void split_nt_core(int M_, int N_, int Kp_, const typename CF::FMT::E *__restrict__ Ap_,
                                                       long a_plane_, int Mp_, const typename CF::FMT::E *__restrict__ Bp_,
                                                       long b_plane_, int Np_, float alpha_, float beta_,
                                                       float *__restrict__ C_, long ldc_, int tiles_m, int tiles_n,
                                                       const unsigned *__restrict__ amax_a_,
                                                       const unsigned *__restrict__ amax_b_, Epilogue epi,
                                                       const float *__restrict__ Af, long lda,
                                                       const float *__restrict__ Bf_, long ldb_, int K_,
                                                       int kt_per, float *__restrict__ ws,
                                                       const GroupedSplitProblem *__restrict__ gprobs,
                                                       const GroupedSplitTile *__restrict__ gtiles) {
    using FMT = typename CF::FMT;
    using E = typename FMT::E;
    using V8 = typename FMT::V8;
    static_assert(!GR || FA == 0, "grouped plans stream A's prepared planes");
    const GroupedSplitTile gt = GR ? gtiles[blockIdx.x] : GroupedSplitTile{0, 0, 0, 0};
    const GroupedSplitProblem *gp = GR ? gprobs + gt.problem : nullptr;
    const int M = GR ? gp->M : M_, N = GR ? gp->N : N_, Kp = GR ? gp->Kp : Kp_;
    const int Mp = GR ? gp->Mp : Mp_, Np = GR ? gp->Np : Np_;
    const E *__restrict__ Ap = GR ? static_cast<const E *>(gp->Ap) : Ap_;
    const E *__restrict__ Bp = GR ? static_cast<const E *>(gp->Bp) : Bp_;
    const long a_plane = GR ? gp->a_plane : a_plane_, b_plane = GR ? gp->b_plane : b_plane_;
    const float alpha = GR ? gp->alpha : alpha_, beta = GR ? gp->beta : beta_;
    float *__restrict__ C = GR ? gp->C : C_;
    const long ldc = GR ? gp->ldc : ldc_;
    const unsigned *__restrict__ amax_a = GR ? gp->amax_a : amax_a_;
    const unsigned *__restrict__ amax_b = GR ? gp->amax_b : amax_b_;
    // B's FP32 source when the core splits it (grouped: per problem).
    const float *__restrict__ Bf = GR ? gp->Bf : Bf_;
    const long ldb = GR ? gp->ldb : ldb_;
    const int K = GR ? gp->K : K_;
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, NP = CF::NP, FM = CF::FM, FN = CF::FN;
    constexpr int CPR = CF::CPR, STAGE = CF::STAGE, STAGES = CF::STAGES, PER_T = CF::PER_T;
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    E *lds = reinterpret_cast<E *>(smem_raw);

    int tm = 0, tn = 0;
    if (!GR) tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = GR ? gt.m0 : tm * BM, n0 = GR ? gt.n0 : tn * BN;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = w / CF::WGN, wn = w % CF::WGN;

    // Stage copy.  In the k-tile blocked plane layout the A tile of K tile kt
    // and plane p is the contiguous block Ap + p*a_plane + (kt*Mp + m0)*BK of
    // BM*BK elements, already in LDS order; likewise B.  Chunk i of thread t
    // is f = t + NT*i (A chunks first), copied to the same position in LDS.
    static_assert(BK == 32, "blocked plane layout uses 32-wide K tiles");
    constexpr int A_CH = NP * BM * CPR / CF::NT;         // 16-byte chunks per thread from A
    static_assert((NP * BM * CPR) % CF::NT == 0 && (BM * CPR) % CF::NT == 0 && (BN * CPR) % CF::NT == 0,
                  "stage split");
    const E *a_src = Ap + (long)m0 * BK + t * 8;
    const E *b_src = Bp + (long)n0 * BK + t * 8;
    constexpr int B_CH = NP * BN * CPR / CF::NT;          // 16-byte chunks per thread from B planes
    constexpr int FA_CH = BM * CPR / CF::NT, FB_CH = BN * CPR / CF::NT;   // fused chunk rows per thread
    static_assert(CPR == 4, "fused staging assumes 32-wide K tiles");
    static_assert((FA != FUSE_RCONT || FA_CH == 1 || FA_CH == 2) && (FB != FUSE_RCONT || FB_CH == 1 || FB_CH == 2),
                  "row-contiguous fusion: one or two rows per thread");
    V8 pa[FA ? 1 : A_CH], pb[FB ? 1 : B_CH];
    float fa[FA ? FA_CH : 1][8], fb[FB ? FB_CH : 1][8];
    // A grouped problem with K == 0 or alpha == 0 (handed over with K = 0) still
    // gets the two K tiles of its zero planes, but has no line of B to read in
    // the place of one past K, and B may be NULL: the stage is zeros, without a
    // load.  Uniform over the block.  A single GEMM never gets here with K == 0.
    const bool no_k = GR && K == 0;
    // Row-contiguous source: rows [r, r+RW) of k-lines k .. k+7 into v[i][j]
    // (row r+i, k+j).  RW is 1 or 2 (stage rows per thread).  Rows past the
    // last read it in their place, without a branch: nothing stores their
    // results.  kin: the stage ends inside K (uniform); else values past K are 0
    // (K >= 1: the last line of K is read in their place).
    // (Guards on rows and k, a branch and a wait each, made the tiles at the
    // edge up to twice as long: 32767x512x1024 TN BF16X3 took 225 us, now 117.)
    auto load_rc = [&](const float *X, long ld, int rows, int r, int k, auto &v, bool kin) {
        constexpr int RW = std::extent<std::remove_reference_t<decltype(v)>>::value;
        const bool pair = RW == 2 && (!GR || rows > 1);   // one problem: run_cfg fuses no single row
        const float *p = X + min(r, rows - (pair ? 2 : 1));   // the last row alone is a pair's second: store_stage
        auto line = [&](const float *q, int j) {
            if (pair) {
                const f32x2u x = *reinterpret_cast<const f32x2u *>(q);
                v[0][j] = x.x;
                v[RW - 1][j] = x.y;
            } else {
                v[0][j] = v[RW - 1][j] = *q;
            }
        };
        if (kin) {
            p += (long)k * ld;
#pragma unroll
            for (int j = 0; j < 8; ++j) line(p + (long)j * ld, j);
        } else if (no_k) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[0][j] = v[RW - 1][j] = 0.0f;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) line(p + (long)min(k + j, K - 1) * ld, j);
#pragma unroll
            for (int i = 0; i < RW; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = k + j < K ? v[i][j] : 0.0f;
        }
    };
    // 8 floats of row `row`, k in [k, k+8), likewise.
    auto load8 = [&](const float *X, long ld, int rows, int row, int k, float (&v)[8], bool kin) {
        const float *p = X + (long)min(row, rows - 1) * ld;
        if (kin) {
            const f32x4u x0 = *reinterpret_cast<const f32x4u *>(p + k);
            const f32x4u x1 = *reinterpret_cast<const f32x4u *>(p + k + 4);
            v[0] = x0.x; v[1] = x0.y; v[2] = x0.z; v[3] = x0.w; v[4] = x1.x; v[5] = x1.y; v[6] = x1.z; v[7] = x1.w;
        } else if (no_k) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = 0.0f;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float x = p[min(k + j, K - 1)];
                v[j] = k + j < K ? x : 0.0f;
            }
        }
    };
    // Plane copy, chunk c (A chunks first): global -> registers, and
    // registers -> LDS buffer buf.
    auto load_chunk = [&](int kt, int c) {
        if (c < A_CH) {
            const int e = c * CF::NT * 8, p = e / (BM * BK), off = e % (BM * BK);
            pa[c] = *reinterpret_cast<const V8 *>(a_src + p * a_plane + (long)kt * Mp * BK + off);
        } else {
            const int e = (c - A_CH) * CF::NT * 8, p = e / (BN * BK), off = e % (BN * BK);
            pb[c - A_CH] = *reinterpret_cast<const V8 *>(b_src + p * b_plane + (long)kt * Np * BK + off);
        }
    };
    auto store_chunk = [&](int buf, int c) {
        E *a_reg = lds + buf * STAGE, *b_reg = a_reg + NP * CF::A_PLANE;
        if (c < A_CH)
            *reinterpret_cast<V8 *>(a_reg + t * 8 + c * CF::NT * 8) = pa[c];
        else
            *reinterpret_cast<V8 *>(b_reg + t * 8 + (c - A_CH) * CF::NT * 8) = pb[c - A_CH];
    };
    auto load_stage = [&](int kt) {
        const int k0 = kt * BK;
        const bool kin = k0 + BK <= K;
        if constexpr (FA == FUSE_RCONT) {
            load_rc(Af, lda, M, m0 + (t % (BM / FA_CH)) * FA_CH, k0 + (t / (BM / FA_CH)) * 8, fa, kin);
        } else if constexpr (FA == FUSE_KCONT) {
#pragma unroll
            for (int i = 0; i < FA_CH; ++i) {
                const int f = t + CF::NT * i, r = f >> 2, c = (f & 3) ^ ((r >> 1) & 3);
                load8(Af, lda, M, m0 + r, k0 + c * 8, fa[i], kin);
            }
        } else {
#pragma unroll
            for (int i = 0; i < A_CH; ++i) load_chunk(kt, i);
        }
        if constexpr (FB == FUSE_RCONT) {
            load_rc(Bf, ldb, N, n0 + (t % (BN / FB_CH)) * FB_CH, k0 + (t / (BN / FB_CH)) * 8, fb, kin);
        } else if constexpr (FB == FUSE_KCONT) {
#pragma unroll
            for (int i = 0; i < FB_CH; ++i) {
                const int f = t + CF::NT * i, r = f >> 2, c = (f & 3) ^ ((r >> 1) & 3);
                load8(Bf, ldb, N, n0 + r, k0 + c * 8, fb[i], kin);
            }
        } else {
#pragma unroll
            for (int i = 0; i < B_CH; ++i) load_chunk(kt, A_CH + i);
        }
    };
    // Scaled formats: the exponents of this thread's fused rows, read once (at
    // each stage, past a barrier, the load stood in front of the split).
    int ea[FA ? FA_CH : 1], eb[FB ? FB_CH : 1];
    bool row_inf = false;   // of any of the wave's fused rows
    auto scales = [&](const unsigned *amax, int mode, int ch, int rows, int r0, auto &e) {
#pragma unroll
        for (int i = 0; i < ch; ++i) {
            const unsigned bits = amax[r0 + (mode == FUSE_RCONT ? (t % (rows / ch)) * ch + i : (t + CF::NT * i) >> 2)];
            e[i] = -row_exp(bits);
            row_inf |= row_is_inf(bits);
        }
    };
    if constexpr (FMT::SCALED && FA != FUSE_NONE) scales(amax_a, FA, FA_CH, BM, m0, ea);
    if constexpr (FMT::SCALED && FB != FUSE_NONE) scales(amax_b, FB, FB_CH, BN, n0, eb);
    if constexpr (FMT::SCALED) row_inf = __any(row_inf);
    // Split one fused chunk (scaled formats: times 2^e) into its NP plane
    // chunks at plane offset f * 8 of the operand's LDS region.
    auto store_fused = [&](E *region, int plane, int e, int f, float (&v)[8]) {
        if constexpr (FMT::SCALED) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = ldexpf(v[j], e);
        }
        V8 w[NP];
        split8<NP, FMT>(v, FMT::SCALED ? row_inf : __any(split_special(FMT(), v, false)), w);
#pragma unroll
        for (int p = 0; p < NP; ++p) *reinterpret_cast<V8 *>(region + p * plane + f * 8) = w[p];
    };
    auto store_stage = [&](int buf) {
        E *a_reg = lds + buf * STAGE, *b_reg = a_reg + NP * CF::A_PLANE;
        if constexpr (FA == FUSE_RCONT) {
            if (FA_CH == 2 && (M & 1) && m0 + BM > M) {   // uniform: the tile at the edge of odd rows
                const bool last = m0 + (t % (BM / FA_CH)) * FA_CH == M - 1;
#pragma unroll
                for (int j = 0; j < 8; ++j) fa[0][j] = last ? fa[FA_CH - 1][j] : fa[0][j];
            }
#pragma unroll
            for (int i = 0; i < FA_CH; ++i) {
                const int r = (t % (BM / FA_CH)) * FA_CH + i, f = r * 4 + ((t / (BM / FA_CH)) ^ ((r >> 1) & 3));
                store_fused(a_reg, CF::A_PLANE, FMT::SCALED ? ea[i] : 0, f, fa[i]);
            }
        } else if constexpr (FA == FUSE_KCONT) {
#pragma unroll
            for (int i = 0; i < FA_CH; ++i) {
                const int f = t + CF::NT * i;
                store_fused(a_reg, CF::A_PLANE, FMT::SCALED ? ea[i] : 0, f, fa[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < A_CH; ++i) store_chunk(buf, i);
        }
        if constexpr (FB == FUSE_RCONT) {
            if (FB_CH == 2 && (N & 1) && n0 + BN > N) {   // uniform: the tile at the edge of odd rows
                const bool last = n0 + (t % (BN / FB_CH)) * FB_CH == N - 1;
#pragma unroll
                for (int j = 0; j < 8; ++j) fb[0][j] = last ? fb[FB_CH - 1][j] : fb[0][j];
            }
#pragma unroll
            for (int i = 0; i < FB_CH; ++i) {
                const int r = (t % (BN / FB_CH)) * FB_CH + i, f = r * 4 + ((t / (BN / FB_CH)) ^ ((r >> 1) & 3));
                store_fused(b_reg, CF::B_PLANE, FMT::SCALED ? eb[i] : 0, f, fb[i]);
            }
        } else if constexpr (FB == FUSE_KCONT) {
#pragma unroll
            for (int i = 0; i < FB_CH; ++i) {
                const int f = t + CF::NT * i;
                store_fused(b_reg, CF::B_PLANE, FMT::SCALED ? eb[i] : 0, f, fb[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < B_CH; ++i) store_chunk(buf, A_CH + i);
        }
    };

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // K tiles [kt0, ktiles) of this block: all of them, or (split-K,
    // gridDim.y > 1) the kt_per tiles of split blockIdx.y, whose alpha = 1,
    // beta = 0 product goes to the partial slice ws + z*M*N (row length N).
    const bool part = gridDim.y > 1;
    const int kt0 = part ? (int)blockIdx.y * kt_per : 0;
    const int ktiles = part ? min(Kp / BK, kt0 + kt_per) : Kp / BK;
    float *const Co = part ? ws + (long)blockIdx.y * M * N : C;
    const long ldo = part ? (long)N : ldc;
    const float al = part ? 1.0f : alpha, be = part ? 0.0f : beta;
    constexpr bool ILV = CF::ILV && !FA && !FB;
    // Fused operands on two stages (ESTORE): stage kt+1, loaded during step
    // kt-1, is split into the idle buffer at the top of step kt and stage
    // kt+2 is loaded right after, so the FP32 loads get a whole step of
    // latency and the split of one block overlaps the MFMAs of others
    // (split at the end of the step, every wave waited on its loads and then
    // split in front of the barrier).  Branch-free like ILV: the last steps
    // store into the idle buffer and re-load the last stage.
    constexpr bool ESTORE = !ILV && (FA || FB) && STAGES == 2;
    load_stage(kt0);
    store_stage(0);
    if constexpr (ILV || ESTORE) load_stage(min(kt0 + 1, ktiles - 1));
    __syncthreads();

    const int frow = lane & 15, fc = lane >> 4;
    if constexpr (CF::EARLY && ILV) {
        // Group (q, i): the FN MFMAs of product q with A fragment i.  In the
        // products before the last, a group reads the A fragment of group
        // (q, i + LA) and (last FN groups) a B fragment of product q + 1, and
        // takes its share of the stage copy (K tile kt + 1 into the idle
        // buffer, K tile kt + 2 into registers).  The barrier then opens the
        // last product, whose planes are held in registers; its groups read
        // K tile kt + 1's first B and A fragments from the other buffer.
        // Every wave has finished reading a buffer (the products before the
        // barrier) before any wave writes it again (after the next barrier).
        constexpr int NQ = Products<NP>::N, LA = 2, NCH = A_CH + B_CH, NGC = (NQ - 1) * FM;
        constexpr int a0 = Products<NP>::a[0], b0 = Products<NP>::b[0];
        static_assert(!first_use_a<NP>(NQ - 1) && !first_use_b<NP>(NQ - 1), "last product from registers");
        V8 fa[NP][FM], fb[NP][FN], na[LA], nb[FN];
        auto frag = [&](const E *base, int row) {
            return *reinterpret_cast<const V8 *>(base + row * BK + swz_chunk<CPR>(row, fc) * 8);
        };
        auto a_row = [&](int i) { return wm * CF::WTM + i * 16 + frow; };
        auto b_row = [&](int j) { return wn * CF::WTN + j * 16 + frow; };
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[b0][j] = frag(lds + NP * CF::A_PLANE + b0 * CF::B_PLANE, b_row(j));
#pragma unroll
        for (int i = 0; i < LA; ++i) fa[a0][i] = frag(lds + a0 * CF::A_PLANE, a_row(i));
        for (int kt = kt0; kt < ktiles; ++kt) {
            const int buf = (kt - kt0) & 1;
            const E *as = lds + buf * STAGE, *bs = as + NP * CF::A_PLANE;
            const E *an = lds + (buf ^ 1) * STAGE, *bn = an + NP * CF::A_PLANE;
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                constexpr int qa = Products<NP>::a[q], qb = Products<NP>::b[q];
                constexpr bool last = q == NQ - 1;
                constexpr int qn = last ? q : q + 1;
                static_for<FM>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (!last) {
                        if constexpr (i + LA < FM) {
                            if constexpr (first_use_a<NP>(q)) fa[qa][i + LA] = frag(as + qa * CF::A_PLANE, a_row(i + LA));
                        } else if constexpr (first_use_a<NP>(qn)) {
                            constexpr int pn = Products<NP>::a[qn];
                            fa[pn][i + LA - FM] = frag(as + pn * CF::A_PLANE, a_row(i + LA - FM));
                        }
                        if constexpr (first_use_b<NP>(qn) && i >= FM - FN) {
                            constexpr int pn = Products<NP>::b[qn];
                            fb[pn][i - (FM - FN)] = frag(bs + pn * CF::B_PLANE, b_row(i - (FM - FN)));
                        }
                        static_for<NCH>([&](auto cc) {
                            constexpr int c = decltype(cc)::value;
                            if constexpr (c * NGC / NCH == q * FM + i) {
                                store_chunk(buf ^ 1, c);
                                load_chunk(min(kt + 2, ktiles - 1), c);
                            }
                        });
                    } else {
                        if constexpr (i == 0) {
                            __syncthreads();
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        if constexpr (i < FN) nb[i] = frag(bn + b0 * CF::B_PLANE, b_row(i));
                        else if constexpr (i - FN < LA) na[i - FN] = frag(an + a0 * CF::A_PLANE, a_row(i - FN));
                    }
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = FMT::mfma(fa[qa][i], fb[qb][j], acc[i][j]);
                });
            });
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[b0][j] = nb[j];
#pragma unroll
            for (int i = 0; i < LA; ++i) fa[a0][i] = na[i];
        }
    } else
    for (int kt = kt0; kt < ktiles; ++kt) {
        const int buf = (STAGES == 2) ? ((kt - kt0) & 1) : 0;
        const bool more = kt + 1 < ktiles;
        if constexpr (ESTORE) {
            store_stage(buf ^ 1);
            load_stage(min(kt + 2, ktiles - 1));
        } else if (!ILV && more) {
            load_stage(kt + 1);
        }
        const E *as = lds + buf * STAGE;
        const E *bs = as + NP * CF::A_PLANE;
#pragma unroll
        for (int s = 0; s < CF::KSTEPS; ++s) {
            V8 fa[NP][FM], fb[NP][FN];
            if constexpr (CF::STREAM && ILV) {
                // Group (q, i): the FN MFMAs of product q with A fragment i.
                // Before its MFMAs a group reads the A fragment that group
                // (q, i + LA) needs (product q + 1's first ones near the end
                // of q), and each of the last FN groups of product q one B
                // fragment of product q + 1.  Planes used again later stay in
                // registers.  A scheduling barrier around every group keeps
                // the reads in this order; the last product deals the stage
                // copy out one chunk per group.
                constexpr int NQ = Products<NP>::N, LA = 2, NCH = A_CH + B_CH;
                auto read_a = [&](int p, int i) {
                    const int row = wm * CF::WTM + i * 16 + frow;
                    fa[p][i] = *reinterpret_cast<const V8 *>(as + p * CF::A_PLANE + row * BK +
                                                             swz_chunk<CPR>(row, s * 4 + fc) * 8);
                };
                auto read_b = [&](int p, int j) {
                    const int row = wn * CF::WTN + j * 16 + frow;
                    fb[p][j] = *reinterpret_cast<const V8 *>(bs + p * CF::B_PLANE + row * BK +
                                                             swz_chunk<CPR>(row, s * 4 + fc) * 8);
                };
#pragma unroll
                for (int j = 0; j < FN; ++j) read_b(Products<NP>::b[0], j);
#pragma unroll
                for (int i = 0; i < LA; ++i) read_a(Products<NP>::a[0], i);
                static_for<NQ>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    constexpr int qa = Products<NP>::a[q], qb = Products<NP>::b[q];
                    constexpr bool last = q == NQ - 1;
                    constexpr int qn = last ? q : q + 1;
                    static_for<FM>([&](auto ic) {
                        constexpr int i = decltype(ic)::value;
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (i + LA < FM) {
                            if constexpr (first_use_a<NP>(q)) read_a(qa, i + LA);
                        } else if constexpr (!last && first_use_a<NP>(qn)) {
                            read_a(Products<NP>::a[qn], i + LA - FM);
                        }
                        if constexpr (!last && first_use_b<NP>(qn) && i >= FM - FN)
                            read_b(Products<NP>::b[qn], i - (FM - FN));
                        if constexpr (last) {
                            // Chunks c with c * FM / NCH == i: store into the
                            // idle buffer, then load stage kt + 2 (the last
                            // steps re-load the last stage: addresses in range).
                            static_for<NCH>([&](auto cc) {
                                constexpr int c = decltype(cc)::value;
                                if constexpr (c * FM / NCH == i) {
                                    store_chunk(buf ^ 1, c);
                                    load_chunk(min(kt + 2, ktiles - 1), c);
                                }
                            });
                        }
#pragma unroll
                        for (int j = 0; j < FN; ++j) acc[i][j] = FMT::mfma(fa[qa][i], fb[qb][j], acc[i][j]);
                    });
                });
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            if constexpr (CF::PHASED) {
                static_for<Products<NP>::N>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    constexpr int pa = Products<NP>::a[q], pb = Products<NP>::b[q];
                    if constexpr (q > 0 && (first_use_a<NP>(q) || first_use_b<NP>(q)))
                        __builtin_amdgcn_sched_barrier(0);
                    if constexpr (first_use_a<NP>(q)) {
#pragma unroll
                        for (int i = 0; i < FM; ++i) {
                            const int row = wm * CF::WTM + i * 16 + frow;
                            fa[pa][i] = *reinterpret_cast<const V8 *>(as + pa * CF::A_PLANE + row * BK +
                                                                      swz_chunk<CPR>(row, s * 4 + fc) * 8);
                        }
                    }
                    if constexpr (first_use_b<NP>(q)) {
#pragma unroll
                        for (int j = 0; j < FN; ++j) {
                            const int row = wn * CF::WTN + j * 16 + frow;
                            fb[pb][j] = *reinterpret_cast<const V8 *>(bs + pb * CF::B_PLANE + row * BK +
                                                                      swz_chunk<CPR>(row, s * 4 + fc) * 8);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j) acc[i][j] = FMT::mfma(fa[pa][i], fb[pb][j], acc[i][j]);
                });
                continue;
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) {
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const int row = wm * CF::WTM + i * 16 + frow;
                    fa[p][i] = *reinterpret_cast<const V8 *>(as + p * CF::A_PLANE + row * BK +
                                                                 swz_chunk<CPR>(row, s * 4 + fc) * 8);
                }
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int row = wn * CF::WTN + j * 16 + frow;
                    fb[p][j] = *reinterpret_cast<const V8 *>(bs + p * CF::B_PLANE + row * BK +
                                                                 swz_chunk<CPR>(row, s * 4 + fc) * 8);
                }
            }
#pragma unroll
            for (int q = 0; q < Products<NP>::N; ++q)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = FMT::mfma(fa[Products<NP>::a[q]][i], fb[Products<NP>::b[q]][j], acc[i][j]);
        }
        if (STAGES == 1) __syncthreads();
        if (!ILV && !ESTORE && more) store_stage(STAGES == 2 ? (buf ^ 1) : 0);
        __syncthreads();
    }

    // Epilogue: C = alpha * acc (+ beta * C), rows 4*(l/16)+r, column l%16 of each fragment;
    // scaled formats first undo the row and column scales: acc * 2^(e_m + e_n).
    // C is read in batches of IB x JB fragments (64 values per lane), all
    // loaded before any is stored: a load cannot move above a store to C
    // that might alias it, so every batch exposes one memory latency.  With
    // 256 accumulators per lane there is no room for a batch (it spills),
    // nor with 16 waves: those variants interleave.
    const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
    const bool has_epi = !GR && !part && epi.active();
    constexpr bool BATCH = FM * FN * 4 < 256;
    constexpr int JB = !BATCH ? 1 : (CF::NT >= 1024 ? 1 : FN);
    constexpr int IB = (JB < FN) ? 1 : (64 / (4 * FN) < 1 ? 1 : (64 / (4 * FN) > FM ? FM : 64 / (4 * FN)));
    static_assert(FM % IB == 0, "whole batches of fragment rows");
#pragma unroll
    for (int i0 = 0; i0 < FM; i0 += IB)
#pragma unroll
    for (int j0 = 0; j0 < FN; j0 += JB) {
        float cv[IB][JB][4];
        if (BATCH && be != 0.0f) {
#pragma unroll
            for (int ii = 0; ii < IB; ++ii) {
                const int mb = m0 + wm * CF::WTM + (i0 + ii) * 16 + (lane >> 4) * 4;
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    const int n = n0 + wn * CF::WTN + (j0 + jj) * 16 + (lane & 15);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        cv[ii][jj][r] = (interior || (mb + r < M && n < N)) ? Co[(long)(mb + r) * ldo + n] : 0.0f;
                }
            }
        }
#pragma unroll
        for (int ii = 0; ii < IB; ++ii) {
            const int i = i0 + ii;
            const int mb = m0 + wm * CF::WTM + i * 16 + (lane >> 4) * 4;
#pragma unroll
            for (int jj = 0; jj < JB; ++jj) {
                const int j = j0 + jj;
                const int n = n0 + wn * CF::WTN + j * 16 + (lane & 15);
                int en = 0;
                if constexpr (FMT::SCALED) en = row_exp(amax_b[n]);   // n < Np: inside the array
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mb + r;
                    if (interior || (m < M && n < N)) {
                        float a = acc[i][j][r];
                        if constexpr (FMT::SCALED) a = ldexpf(a, row_exp(amax_a[m]) + en);
                        float *cp = Co + (long)m * ldo + n;
                        float v = (be == 0.0f) ? al * a : fmaf(al, a, be * (BATCH ? cv[ii][jj][r] : *cp));
                        if (has_epi) v = apply_epilogue(epi, v, m, n);
                        *cp = v;
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Variants: (tile, BK) per form.
template <int NP, class FMT = FmtBf16>
struct Table;
// V0-V3: 4 waves (2 x 2), one per SIMD.  V4, V5: 8 or 16 waves, 2 or 4 per
// SIMD, which hide each other's LDS and global latency (measured at 8192^3:
// 15-20% faster core than V0).  V6: 8 waves with streamed reads, the
// interleaved stage copy and (NP >= 2) the early barrier; 6-10% faster than
// V5 at 8192^3.  NP = 1, 2: 256x256x32 tiles (32 / 64 KiB per stage); NP = 3:
// 256x128x32 (72 KiB per stage).  V7: V6's schedule on 128x128 tiles (8
// waves of 64x32) for grids too small for V6.  Smaller tiles serve small
// grids.
template <>
struct Table<1> {
    using V0 = CoreCfg<256, 256, 32, 1>;
    using V1 = CoreCfg<128, 128, 32, 1>;
    using V2 = CoreCfg<256, 128, 32, 1>;
    using V3 = CoreCfg<64, 64, 32, 1>;
    using V4 = CoreCfg<256, 256, 32, 1, FmtBf16, 2, 4, false>;
    using V5 = CoreCfg<256, 256, 32, 1, FmtBf16, 4, 4, true>;
    using V6 = CoreCfg<256, 256, 32, 1, FmtBf16, 2, 4, true, true, true>;
    using V7 = CoreCfg<128, 128, 32, 1, FmtBf16, 2, 4, true, true, true>;
};
template <>
struct Table<2> {
    using V0 = CoreCfg<256, 256, 32, 2>;
    using V1 = CoreCfg<128, 128, 32, 2>;
    using V2 = CoreCfg<256, 128, 32, 2>;
    using V3 = CoreCfg<64, 64, 32, 2>;
    using V4 = CoreCfg<256, 256, 32, 2, FmtBf16, 2, 4, false>;
    using V5 = CoreCfg<256, 256, 32, 2, FmtBf16, 4, 4, true>;
    using V6 = CoreCfg<256, 256, 32, 2, FmtBf16, 2, 4, true, true, true, true>;
    using V7 = CoreCfg<128, 128, 32, 2, FmtBf16, 2, 4, true, true, true, true>;
};
template <>
struct Table<3> {
    using V0 = CoreCfg<256, 128, 32, 3>;
    using V1 = CoreCfg<128, 128, 32, 3>;
    using V2 = CoreCfg<128, 256, 32, 3>;
    using V3 = CoreCfg<64, 64, 32, 3>;
    using V4 = CoreCfg<256, 128, 32, 3, FmtBf16, 2, 4, true>;
    using V5 = CoreCfg<256, 128, 32, 3, FmtBf16, 4, 2, true>;
    using V6 = CoreCfg<256, 128, 32, 3, FmtBf16, 2, 4, true, true, true, true>;
    using V7 = CoreCfg<128, 128, 32, 3, FmtBf16, 2, 4, true, true, true, true>;
};
template <>
struct Table<2, FmtF16> {
    using V0 = CoreCfg<256, 256, 32, 2, FmtF16>;
    using V1 = CoreCfg<128, 128, 32, 2, FmtF16>;
    using V2 = CoreCfg<256, 128, 32, 2, FmtF16>;
    using V3 = CoreCfg<64, 64, 32, 2, FmtF16>;
    using V4 = CoreCfg<256, 256, 32, 2, FmtF16, 2, 4, false>;
    using V5 = CoreCfg<256, 256, 32, 2, FmtF16, 4, 4, true>;
    using V6 = CoreCfg<256, 256, 32, 2, FmtF16, 2, 4, true, true, true, true>;
    using V7 = CoreCfg<128, 128, 32, 2, FmtF16, 2, 4, true, true, true, true>;
};
constexpr int kNumVariants = 8;

template <class CF>
const char *cfg_name() {
    // Formatted once per instantiation; function-local static initialisation is thread-safe.
    static const std::string name = [] {
        char buf[48];
        snprintf(buf, sizeof buf, "%sx%d_nt_%dx%dx%d_w%dx%d%s", CF::FMT::name,
                 CF::NP == 1 ? 1 : (CF::NP == 2 ? 3 : 6), CF::BM, CF::BN, CF::BK, CF::WGM, CF::WGN,
                 CF::EARLY ? "_st_early" : (CF::STREAM ? "_st" : (CF::PHASED ? "_ph" : "")));
        return std::string(buf);
    }();
    return name.c_str();
}

int planes_of(int mode) {
    switch (mode) {
        case UGEMM_MODE_BF16X1: return 1;
        case UGEMM_MODE_BF16X3: return 2;
        case UGEMM_MODE_BF16X6: return 3;
        case UGEMM_MODE_FP16X3: return 2;
        default: return 0;
    }
}

static long round_up(long x, long a) { return (x + a - 1) / a * a; }

// One operand of a GEMM to prepare: its source, its planes (out null: the core
// splits it, only the row maxima are wanted), row maxima (scaled formats) and,
// if there is room for them, partial maxima (kAmaxParts rows of rows_pad).
struct Side {
    const float *X;
    long ld;
    bool kcont;
    int rows, rows_pad;
    void *out;
    long plane_stride;
    unsigned *amax, *parts;
};
bool side_in_parts(bool kcont, bool planes, int K) {
    return !kcont && planes && (K + kAmaxRcontSpan - 1) / kAmaxRcontSpan <= kAmaxParts;
}

// Planes and row maxima of up to two operands in the fewest launches, each
// 4-5 us of a call: the BF16 forms one.  FP16X3 one where every operand is
// k-contiguous with K <= 8192 (row maximum and split of whole rows together);
// else the maxima of both (or the whole rows of one) in one and the remaining
// planes in another.  Row-contiguous operands with K <= 2048 hand partial
// maxima over; longer ones, and those split in the core, combine them in
// memory, which a fill clears first (a kernel, not a memset: callers may capture
// this call in a graph).
// us a call, one preparation an operand and a fill before / now: 655x4518x667 TN
// 68 / 43, 543x128x3603 TT 46 / 34, 700x3000x1000 NN 52 / 46, 2048^3 NT 79 / 76.
template <int NP, class FMT>
int prep_operands(Side a, Side b, int K, int k_pad, bool zeroed, hipStream_t s) {
    bool rows_done[2] = {false, false};
    Side *sides[2] = {&a, &b};
    if constexpr (FMT::SCALED) {
        ScaleJob jobs[2] = {};
        bool combine = false;
        for (int i = 0; i < 2; ++i) {
            Side &d = *sides[i];
            ScaleJob &j = jobs[i];
            if (!d.X) continue;
            j.X = d.X;
            j.ld = d.ld;
            j.plane_stride = d.plane_stride;
            j.out = d.out;
            j.amax = d.amax;
            j.parts = d.parts;
            j.rows = d.rows;
            j.rows_pad = d.rows_pad;
            j.k_pad = k_pad;
            long blocks;
            if (d.kcont && d.out && k_pad <= 8192) {
                j.kind = SCALE_SPLIT_ROWS;
                j.chunks = row_lanes(k_pad);
                blocks = d.rows_pad / (512 / j.chunks);
                rows_done[i] = true;
            } else if (d.kcont) {
                j.kind = SCALE_KCONT;
                j.chunks = (K + 2047) / 2048;
                blocks = j.chunks == 1 ? d.rows_pad : d.rows * j.chunks;
                combine |= j.chunks > 1;
            } else {
                const long kblocks = (K + kAmaxRcontSpan - 1) / kAmaxRcontSpan;
                const bool parts = d.parts != nullptr, narrow = kblocks * ((d.rows + 255) / 256) < device_cu_count();
                j.kind = parts ? (narrow ? SCALE_PARTS_NARROW : SCALE_PARTS) : (narrow ? SCALE_RCONT_NARROW : SCALE_RCONT);
                blocks = kblocks * (narrow ? (d.rows + 63) / 64 : (d.rows + 255) / 256);
                combine |= !parts;
            }
            if (blocks > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "too many row blocks");
            j.blocks = (int)blocks;
        }
        if (combine && !zeroed)   // the maxima of both operands, one array
            hipLaunchKernelGGL(fill_zero_u32, dim3((unsigned)std::min<long>((a.rows_pad + b.rows_pad + 255) / 256, 1024)),
                               dim3(256), 0, s, a.amax, (long)a.rows_pad + b.rows_pad);
        // The scans first: whole rows keep a block busier.
        const bool swap = jobs[0].kind == SCALE_SPLIT_ROWS;
        const long blocks = (long)jobs[0].blocks + jobs[1].blocks;
        if (blocks > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "too many row blocks");
        hipLaunchKernelGGL((split_scales<NP, FMT>), dim3((unsigned)blocks), dim3(256), 0, s, jobs[swap], jobs[!swap], K);
    }
    PrepJob jobs[2] = {};
    long blocks = 0;
    for (int i = 0; i < 2; ++i) {
        const Side &d = *sides[i];
        PrepJob &j = jobs[i];
        j.block0 = (int)blocks;
        if (!d.X || !d.out || rows_done[i]) continue;
        j.X = d.X;
        j.ld = d.ld;
        j.out = d.out;
        j.plane_stride = d.plane_stride;
        j.rows = d.rows;
        j.K = K;
        j.rows_pad = d.rows_pad;
        j.k_pad = k_pad;
        j.kcont = d.kcont;
        j.nbx = d.rows_pad / 64;
        j.amax = d.amax;
        j.parts = d.parts;
        j.nparts = d.parts ? (K + kAmaxRcontSpan - 1) / kAmaxRcontSpan : 0;
        blocks += (long)j.nbx * (d.kcont ? (k_pad + 127) / 128 : k_pad / 64);
        if (blocks > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "too many preparation blocks");
    }
    if (blocks > 0)
        hipLaunchKernelGGL((split_prep_pair<NP, FMT>), dim3((unsigned)blocks), dim3(256), 0, s, jobs[0], jobs[1]);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? UGEMM_OK : hip_fail(e, "split preparation");
}

// Split-K count of the core's grid, with *kc the K chunk (whole 32-wide K tiles).
template <class CF>
int core_splits(const Gemm<float> &g, int tiles_m, int tiles_n, int Kp, int *kc) {
    *kc = Kp;
    return split_count(g.splits, (long)tiles_m * tiles_n, Kp, CF::BK, kc, CF::NT >= 512 ? 1 : 2);
}

// The core launch (and, split along K, the reduction of the partial products
// in ws, splits * M * N floats that the caller allocated with the planes).
template <class CF, int FA, int FB>
int launch_core(const Gemm<float> &g, const typename CF::FMT::E *Ap, long a_plane, int Mp, const typename CF::FMT::E *Bp,
                long b_plane, int Np, int Kp, int tiles_m, int tiles_n, const unsigned *amax_a,
                const unsigned *amax_b, int splits, int kc, float *ws, hipStream_t s) {
    auto kern = split_nt_core<CF, FA, FB>;
    // Once per kernel instantiation (thread-safe static initialisation).
    static const hipError_t attr = hipFuncSetAttribute((const void *)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, CF::LDS_BYTES);
    if (attr != hipSuccess) return hip_fail(attr, "hipFuncSetAttribute");
    timing_begin(s);
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n), (unsigned)splits), dim3(CF::NT), CF::LDS_BYTES, s,
                       g.M, g.N, Kp, Ap, a_plane, Mp, Bp, b_plane, Np, g.alpha, g.beta, g.C, g.ldc, tiles_m, tiles_n,
                       amax_a, amax_b, g.epi, g.A, g.lda, g.B, g.ldb, g.K, kc / CF::BK, ws,
                       (const GroupedSplitProblem *)nullptr, (const GroupedSplitTile *)nullptr);
    timing_end(s);
    hipError_t e = hipGetLastError();
    int rc = e == hipSuccess ? UGEMM_OK : hip_fail(e, "split core launch");
    if (!rc && splits > 1) rc = launch_splitk_reduce_f32(g.M, g.N, splits, g.alpha, ws, g.beta, g.C, g.ldc, g.epi, s);
    return rc;
}

// One workspace per call, allocated before the first launch: the planes and
// row maxima (base_bytes, then 256 bytes of slack), then the split-K partial
// products at the next 256-byte boundary.
static size_t splitk_ws_offset(size_t base_bytes) { return (base_bytes + 256 + 255) / 256 * 256; }
static size_t splitk_ws_bytes(int splits, const Gemm<float> &g) {
    return splits > 1 ? (size_t)splits * g.M * g.N * sizeof(float) : 0;
}

// Workspace: NP planes of A (Mp x Kp) and of B (Np x Kp) -- none for an
// operand the core splits itself -- then (scaled formats) Mp + Np row maxima.
template <class CF>
int run_cfg(const Gemm<float> &g, hipStream_t s) {
    using FMT = typename CF::FMT;
    using E = typename FMT::E;
    constexpr int NP = CF::NP;
    const long Mp = round_up(g.M, CF::BM), Np = round_up(g.N, CF::BN), Kp = round_up(g.K, 64);
    // A k-contiguous FP32 source (A not transposed, B transposed) read by at
    // most two tiles along the other dimension is split in the core (8-wave
    // variants): its preparation pass would cost as much as the GEMM reads.
    // Operands re-read by many tiles stay on prepared planes, whose blocked
    // layout the core streams contiguously (measured: splitting a re-read
    // operand in the core is ~50% slower at 8192^3).
    // A row-contiguous source (A transposed, B not) is transposed in
    // registers on the way; that needs one or two rows per thread.  At most one
    // operand is fused per call (the larger, when both qualify).
    constexpr int RW_A = CF::BM * CF::CPR / CF::NT, RW_B = CF::BN * CF::CPR / CF::NT;
    constexpr bool RC_A = RW_A == 1 || RW_A == 2, RC_B = RW_B == 1 || RW_B == 2;
    bool fa = CF::FUSABLE && Np / CF::BN <= 2 && (!g.ta || (RC_A && g.M >= RW_A));
    bool fb = CF::FUSABLE && Mp / CF::BM <= 2 && (g.tb || (RC_B && g.N >= RW_B));
    if (fa && fb) (g.M >= g.N ? fb : fa) = false;
    const int fa_mode = !fa ? FUSE_NONE : (g.ta ? FUSE_RCONT : FUSE_KCONT);
    const int fb_mode = !fb ? FUSE_NONE : (g.tb ? FUSE_KCONT : FUSE_RCONT);
    const long a_plane = Mp * Kp, b_plane = Np * Kp;
    const size_t a_bytes = fa ? 0 : (size_t)NP * a_plane * sizeof(E), b_bytes = fb ? 0 : (size_t)NP * b_plane * sizeof(E);
    const size_t amax_bytes = FMT::SCALED ? (size_t)(Mp + Np) * sizeof(unsigned) : 0;
    const int tiles_m = (int)(Mp / CF::BM), tiles_n = (int)(Np / CF::BN);
    if ((long)tiles_m * tiles_n > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "too many tiles");
    if (FMT::SCALED && (long)g.M * ((g.K + 2047) / 2048) > 0x7fffffffL)
        return fail(UGEMM_ERR_ARG, "too many row blocks");
    int kc;
    const int splits = core_splits<CF>(g, tiles_m, tiles_n, (int)Kp, &kc);
    // Partial maxima only where they don't take the call beyond the scratch of
    // the no-allocation entry.
    const size_t base = a_bytes + b_bytes + amax_bytes, sums = splitk_ws_bytes(splits, g);
    size_t a_parts = FMT::SCALED && side_in_parts(!g.ta, !fa, g.K) ? (size_t)kAmaxParts * Mp * sizeof(unsigned) : 0;
    size_t b_parts = FMT::SCALED && side_in_parts(g.tb, !fb, g.K) ? (size_t)kAmaxParts * Np * sizeof(unsigned) : 0;
    if (splitk_ws_offset(base) + sums <= UGEMM_HIP_NOALLOC_SCRATCH_BYTES &&
        splitk_ws_offset(base + a_parts + b_parts) + sums > UGEMM_HIP_NOALLOC_SCRATCH_BYTES)
        a_parts = b_parts = 0;
    const size_t ws_off = splitk_ws_offset(base + a_parts + b_parts);
    void *ws = nullptr;
    int rc = stream_alloc(&ws, ws_off + sums, s);
    if (rc) return rc;
    E *Ap = (E *)ws, *Bp = (E *)((char *)ws + a_bytes);
    unsigned *amax_a = FMT::SCALED ? (unsigned *)((char *)ws + a_bytes + b_bytes) : nullptr;
    unsigned *amax_b = FMT::SCALED ? amax_a + Mp : nullptr;
    unsigned *parts_a = a_parts ? (unsigned *)((char *)ws + base) : nullptr;
    unsigned *parts_b = b_parts ? (unsigned *)((char *)ws + base + a_parts) : nullptr;
    float *part = splits > 1 ? (float *)((char *)ws + ws_off) : nullptr;
    const Side sa = {g.A, g.lda, !g.ta, g.M, (int)Mp, fa ? nullptr : Ap, a_plane, amax_a, parts_a};
    const Side sb = {g.B, g.ldb, (bool)g.tb, g.N, (int)Np, fb ? nullptr : Bp, b_plane, amax_b, parts_b};
    // The BF16 forms need nothing of an operand that the core splits.
    if (FMT::SCALED || !fa || !fb)
        rc = prep_operands<NP, FMT>(sa, sb, g.K, (int)Kp, false, s);
    if (!rc) {
        const unsigned *ma = amax_a, *mb = amax_b;
#define UGEMM_CORE(FA_, FB_) \
    launch_core<CF, FA_, FB_>(g, Ap, a_plane, (int)Mp, Bp, b_plane, (int)Np, (int)Kp, tiles_m, tiles_n, ma, mb, splits, \
                              kc, part, s)
        if constexpr (CF::FUSABLE) {
            if (fa_mode == FUSE_KCONT) rc = UGEMM_CORE(FUSE_KCONT, FUSE_NONE);
            else if (fb_mode == FUSE_KCONT) rc = UGEMM_CORE(FUSE_NONE, FUSE_KCONT);
            else if (fa_mode == FUSE_RCONT) {
                if constexpr (RC_A) rc = UGEMM_CORE(FUSE_RCONT, FUSE_NONE);
            } else if (fb_mode == FUSE_RCONT) {
                if constexpr (RC_B) rc = UGEMM_CORE(FUSE_NONE, FUSE_RCONT);
            } else rc = UGEMM_CORE(FUSE_NONE, FUSE_NONE);
        } else {
            rc = UGEMM_CORE(FUSE_NONE, FUSE_NONE);
        }
#undef UGEMM_CORE
    }
    int rc2 = stream_free(ws, s);
    return rc ? rc : rc2;
}

template <int NP, class FMT = FmtBf16>
int launch_np(const Gemm<float> &g, int variant, hipStream_t s) {
    using T = Table<NP, FMT>;
    switch (variant) {
        case 0: return run_cfg<typename T::V0>(g, s);
        case 1: return run_cfg<typename T::V1>(g, s);
        case 2: return run_cfg<typename T::V2>(g, s);
        case 3: return run_cfg<typename T::V3>(g, s);
        case 4: return run_cfg<typename T::V4>(g, s);
        case 5: return run_cfg<typename T::V5>(g, s);
        case 6: return run_cfg<typename T::V6>(g, s);
        case 7: return run_cfg<typename T::V7>(g, s);
        default: return fail(UGEMM_ERR_ARG, "split form: no variant %d", variant);
    }
}

// Convolution as a split-form GEMM: C (channels x pixels) = weights (M x K,
// k-contiguous) times the im2col operand, whose planes are gathered from the
// image by split_prep_im2col; then the core with the epilogue.
template <class CF>
int run_cfg_conv(const Gemm<float> &g, const ConvDesc &cd, hipStream_t s) {
    using FMT = typename CF::FMT;
    using E = typename FMT::E;
    constexpr int NP = CF::NP;
    const long Mp = round_up(g.M, CF::BM), Np = round_up(g.N, CF::BN), Kp = round_up(g.K, 64);
    const long a_plane = Mp * Kp, b_plane = Np * Kp;
    const size_t a_bytes = (size_t)NP * a_plane * sizeof(E), b_bytes = (size_t)NP * b_plane * sizeof(E);
    const size_t amax_bytes = FMT::SCALED ? (size_t)(Mp + Np) * sizeof(unsigned) : 0;
    const int tiles_m = (int)(Mp / CF::BM), tiles_n = (int)(Np / CF::BN);
    if ((long)tiles_m * tiles_n > 0x7fffffffL) return fail(UGEMM_ERR_ARG, "too many tiles");
    if (FMT::SCALED && (long)g.M * ((g.K + 2047) / 2048) > 0x7fffffffL)
        return fail(UGEMM_ERR_ARG, "too many row blocks");
    int kc;
    const int splits = core_splits<CF>(g, tiles_m, tiles_n, (int)Kp, &kc);
    const size_t ws_off = splitk_ws_offset(a_bytes + b_bytes + amax_bytes);
    void *ws = nullptr;
    int rc = stream_alloc(&ws, ws_off + splitk_ws_bytes(splits, g), s);
    if (rc) return rc;
    E *Ap = (E *)ws, *Bp = (E *)((char *)ws + a_bytes);
    unsigned *amax_a = FMT::SCALED ? (unsigned *)((char *)ws + a_bytes + b_bytes) : nullptr;
    unsigned *amax_b = FMT::SCALED ? amax_a + Mp : nullptr;
    float *part = splits > 1 ? (float *)((char *)ws + ws_off) : nullptr;
    if (FMT::SCALED)
        hipLaunchKernelGGL(fill_zero_u32, dim3((unsigned)std::min<long>((Mp + Np + 255) / 256, 1024)), dim3(256), 0,
                           s, amax_a, Mp + Np);
    rc = prep_operands<NP, FMT>(Side{g.A, g.lda, true, g.M, (int)Mp, Ap, a_plane, amax_a, nullptr}, Side{}, g.K,
                                (int)Kp, true, s);
    if (!rc) {
        constexpr int KSPAN = 32;   // short spans: enough blocks for small images
        if (FMT::SCALED)
            hipLaunchKernelGGL(row_amax_im2col, dim3((unsigned)((g.N + 255) / 256), (unsigned)((g.K + KSPAN - 1) / KSPAN)),
                               dim3(256), 0, s, cd, g.N, g.K, KSPAN, amax_b);
        const long total = Np * (Kp / 8);
        const long blocks = std::max<long>(1, std::min<long>((total + 255) / 256, 64L * device_cu_count()));
        hipLaunchKernelGGL((split_prep_im2col<NP, FMT>), dim3((unsigned)blocks), dim3(256), 0, s, cd, g.N, g.K, Bp,
                           b_plane, (int)Np, (int)Kp, (const unsigned *)amax_b);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = hip_fail(e, "conv: operand gather");
    }
    if (!rc)
        rc = launch_core<CF, FUSE_NONE, FUSE_NONE>(g, Ap, a_plane, (int)Mp, Bp, b_plane, (int)Np, (int)Kp, tiles_m,
                                                   tiles_n, amax_a, amax_b, splits, kc, part, s);
    const int rc2 = stream_free(ws, s);
    return rc ? rc : rc2;
}

template <int NP, class FMT = FmtBf16>
int launch_np_conv(const Gemm<float> &g, const ConvDesc &cd, int variant, hipStream_t s) {
    using T = Table<NP, FMT>;
    switch (variant) {
        case 0: return run_cfg_conv<typename T::V0>(g, cd, s);
        case 1: return run_cfg_conv<typename T::V1>(g, cd, s);
        case 2: return run_cfg_conv<typename T::V2>(g, cd, s);
        case 3: return run_cfg_conv<typename T::V3>(g, cd, s);
        case 4: return run_cfg_conv<typename T::V4>(g, cd, s);
        case 5: return run_cfg_conv<typename T::V5>(g, cd, s);
        case 6: return run_cfg_conv<typename T::V6>(g, cd, s);
        case 7: return run_cfg_conv<typename T::V7>(g, cd, s);
        default: return fail(UGEMM_ERR_ARG, "split form: no variant %d", variant);
    }
}

template <int NP, class FMT = FmtBf16>
const char *name_np(int v) {
    using T = Table<NP, FMT>;
    switch (v) {
        case 0: return cfg_name<typename T::V0>();
        case 1: return cfg_name<typename T::V1>();
        case 2: return cfg_name<typename T::V2>();
        case 3: return cfg_name<typename T::V3>();
        case 4: return cfg_name<typename T::V4>();
        case 5: return cfg_name<typename T::V5>();
        case 6: return cfg_name<typename T::V6>();
        case 7: return cfg_name<typename T::V7>();
        default: return nullptr;
    }
}

}  // namespace

int mfma_variant_count(int mode) { return planes_of(mode) ? kNumVariants : 0; }

const char *mfma_variant_name(int mode, int v) {
    if (v < 0 || v >= kNumVariants) return nullptr;
    switch (mode) {
        case UGEMM_MODE_BF16X1: return name_np<1>(v);
        case UGEMM_MODE_BF16X3: return name_np<2>(v);
        case UGEMM_MODE_BF16X6: return name_np<3>(v);
        case UGEMM_MODE_FP16X3: return name_np<2, FmtF16>(v);
        default: return nullptr;
    }
}

// The estimate behind the choice on grids of fewer than one 256-row tile a CU,
// in us, fitted to splits 1-16 of variants 3, 7 and the large tile over 31
// shapes (sides 33..15277, K 186..42112; rms 7-11% a form).  The CU with the
// most blocks sets the time: `most` blocks of `us` per 1000 of K, of which
// latency stretches few (`lat`; up to `occ` share a CU), and `block` each for
// the first loads and the epilogue.  Partial sums cost a second launch and
// their bytes, the preparation its bytes (FP16X3 reads an operand twice, once
// for the row maxima), and an operand that the core splits spares it that for
// `fused` times the core.  A copy moves 4.8 bytes a ps.
namespace {
struct PickTile {
    int variant, bm, bn;
    double us, lat, occ, block;
};
struct PickForm {
    PickTile tile[3];
    double prep, fused;
};
const PickForm &pick_form(int np) {
    static const PickForm forms[3] = {
        {{{3, 64, 64, 1.5, 6.0, 4, 0.4}, {7, 128, 128, 8.0, 0.3, 2, 2.0}, {5, 256, 256, 22, 0.1, 1, 12}}, 1.5, 1.9},
        {{{3, 64, 64, 4.4, 1.9, 4, 0.4}, {7, 128, 128, 13.5, 0.3, 2, 2.0}, {6, 256, 256, 43, 0.1, 1, 15}}, 1.8, 1.5},
        {{{3, 64, 64, 8.7, 0.9, 4, 1.2}, {7, 128, 128, 28.0, 0.1, 2, 3.0}, {6, 256, 128, 49, 0.1, 1, 8}}, 2.5, 1.3}};
    return forms[np - 1];
}

// The operand (at most one) that the core splits itself: run_cfg's rule.
void fused_operand(const Gemm<float> &g, int variant, long tm, long tn, bool *fa, bool *fb) {
    const bool eight = variant == 4 || variant == 6 || variant == 7;
    *fa = eight && tn <= 2;
    *fb = eight && tm <= 2;
    if (*fa && *fb) (g.M >= g.N ? *fb : *fa) = false;
}

// Microseconds of g on tile t with S splits; *ws receives the workspace bytes.
double pick_cost(const Gemm<float> &g, int np, bool scaled, bool fusable, const PickForm &f, const PickTile &t, int S,
                 size_t *ws) {
    const double cus = (double)device_cu_count(), per_us = 4.8e6;
    const long tm = (g.M + t.bm - 1) / t.bm, tn = (g.N + t.bn - 1) / t.bn, kc = ((g.K + S - 1) / S + 31) / 32 * 32;
    bool fa = false, fb = false;
    if (fusable) fused_operand(g, t.variant, tm, tn, &fa, &fb);
    const long ra = tm * t.bm, rb = tn * t.bn;
    const double left = scaled ? 0.5 : 0.0;   // of a fused operand's preparation: its row maxima
    const double prep = ((fa ? left : 1.0) * ra + (fb ? left : 1.0) * rb) * g.K;
    const double most = std::ceil(tm * tn * S / cus);
    double us = t.us * (fa || fb ? f.fused : 1.0) * kc / 1000.0 * (1.0 + t.lat / std::min(most, t.occ));
    us = (us + t.block) * most + (scaled ? 2.5 : f.prep) * prep * 4 / per_us;
    const double sums = S > 1 ? 4.0 * S * g.M * g.N : 0.0;
    if (S > 1) us += 2.5 + 0.9 * sums / per_us;
    *ws = ((fa ? 0 : ra) + (fb ? 0 : rb)) * (size_t)round_up(g.K, 64) * 2 * np + (scaled ? (ra + rb) * 4 : 0) + 512 +
          (size_t)sums;
    return us;
}

// What the choice by the grid alone (mfma_fixed_variant) takes: its split count and workspace.
double fixed_cost(const Gemm<float> &g, int np, bool scaled, bool fusable, const PickForm &f, int fixed, size_t *ws) {
    for (const PickTile &t : f.tile) {
        if (t.variant != fixed) continue;
        int kc;
        const long tiles = (long)((g.M + t.bm - 1) / t.bm) * ((g.N + t.bn - 1) / t.bn);
        const int S = split_count(0, tiles, (int)round_up(g.K, 64), 32, &kc, fixed == 3 ? 2 : 1);
        return pick_cost(g, np, scaled, fusable, f, t, S, ws);
    }
    *ws = 0;
    return 0;
}

// Grids of fewer 256-row tiles than CUs, without a split count.  128 x 128
// tiles: the 8-wave streamed V7 (2048^3: 12-24% faster per call than the
// 4-wave V1, whose one wave per SIMD hides no latency).
int mfma_fixed_variant(const Gemm<float> &g) {
    return (long)((g.M + 127) / 128) * ((g.N + 127) / 128) >= device_cu_count() / 2 ? 7 : 3;
}
}  // namespace

bool mfma_planes_fit_scratch(const Gemm<float> &g, int mode) {
    const int np = planes_of(mode);
    for (const int v : {3, mfma_fixed_variant(g)}) {
        size_t ws;
        fixed_cost(g, np, mode == UGEMM_MODE_FP16X3, true, pick_form(np), v, &ws);
        if (ws <= UGEMM_HIP_NOALLOC_SCRATCH_BYTES) return true;
    }
    return false;
}

int mfma_pick_variant(const Gemm<float> &g, int mode, bool fusable, int *splits) {
    const long cus = device_cu_count();
    const int np = planes_of(mode);
    // Largest tile whose grid still gives every CU work; there, the
    // multi-wave variant measured fastest for the form.
    const long big_m = 256, big_n = (np == 3) ? 128 : 256;
    const long tm = (g.M + big_m - 1) / big_m, tn = (g.N + big_n - 1) / big_n;
    // A skinny side whose operand (either layout) the 8-wave variant
    // splits in the core (no preparation pass): V4.  Otherwise two and
    // three planes run fastest on the streamed V6, one plane on the
    // 16-wave V5.
    const int big = fusable && np <= 2 && (tn <= 2 || tm <= 2) ? 4 : (np >= 2 ? 6 : 5);
    if (tm * tn >= cus) {
        // A few tiles more than CUs: the second round is nearly empty, and V7's
        // 128x128 tiles, 1.4 times as dear by area, come out ahead (us, V6 or V5 /
        // V7, 289 tiles: 4200x4200x2048 BF16X3 294 / 244, FP16X3 325 / 262, BF16X1
        // 139 / 129; 360 tiles, 5000x4500x1500 222 / 210, 384 287 / 293).  Not for
        // three planes, whose large tile is half as wide.  Same bits.
        const double t128 = (double)((g.M + 127) / 128) * ((g.N + 127) / 128);
        if (np <= 2 && big != 4 && !stream_alloc_is_static() &&
            1.4 * 0.25 * std::ceil(t128 / cus) < 0.95 * ((tm * tn + cus - 1) / cus))
            return 7;
        return big;
    }
    const int fixed = mfma_fixed_variant(g);
    if (*splits > 0 || g.K <= 0) return fixed;
    // Fewer: tile and splits together.  493x2304x34854 BF16X3 ran 288 blocks
    // of V3 in 877 us, one wave a SIMD and two blocks on a few CUs; V4 in 14
    // splits takes 270.  1024x1024x4096 54 and 47 (V7 in 4), 64x6272x6592 91
    // and 53 (V7 in 8, which splits B in the core), 5120x111x6405 93 and 48.
    // Near ties stay with the fixed choice and its own split count.  What that
    // runs within the scratch of the no-allocation entry stays within it, and
    // there the calls that it refuses stay refused: one choice for both entries.
    const bool scaled = mode == UGEMM_MODE_FP16X3;
    const PickForm &f = pick_form(np);
    size_t ws, fixed_ws;
    double best = 0.92 * fixed_cost(g, np, scaled, fusable, f, fixed, &fixed_ws);
    const bool fits = fixed_ws <= UGEMM_HIP_NOALLOC_SCRATCH_BYTES;
    if (!fits && stream_alloc_is_static()) return fixed;
    int v = fixed;
    for (PickTile t : f.tile) {
        if (t.bm == 256) t.variant = big;
        for (int S = 1; S <= 16 && (S == 1 || (g.K / S >= 256 && (size_t)S * g.M * g.N * 4 <= (64u << 20))); ++S) {
            const double c = pick_cost(g, np, scaled, fusable, f, t, S, &ws);
            if (c < best && (!fits || ws <= UGEMM_HIP_NOALLOC_SCRATCH_BYTES)) {
                best = c;
                v = t.variant;
                *splits = S;
            }
        }
    }
    return v;
}

// ---------------------------------------------------------------------------
// Grouped split-form plans (grouped.hip): any variant, on planes of both
// operands, or those that split B in the core; the FP16 form adds the row-maximum
// pass.
namespace {
template <class CF, int FB = FUSE_NONE>
int grouped_core(const PrepJob *jobs, const int *block_job, int prep_blocks, const GroupedSplitProblem *probs,
                 const GroupedSplitTile *tiles, int ntiles, hipStream_t s, const GroupedScales *sc) {
    using FMT = typename CF::FMT;
    if (FMT::SCALED) {
        // Row maxima first (a fill kernel, not a memset: the launches are captured in graphs).
        hipLaunchKernelGGL(fill_zero_u32, dim3((unsigned)std::min<long>((sc->count + 255) / 256, 4096)), dim3(256), 0,
                           s, sc->amax, sc->count);
        if (sc->blocks > 0)
            hipLaunchKernelGGL(grouped_row_amax, dim3((unsigned)sc->blocks), dim3(256), 0, s, sc->jobs,
                               sc->block_job);
    }
    if (prep_blocks > 0)
        hipLaunchKernelGGL((grouped_split_prep<CF::NP, FMT>), dim3((unsigned)prep_blocks), dim3(256), 0, s, jobs,
                           block_job);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "grouped split-form preparation");
    auto kern = split_nt_core<CF, FUSE_NONE, FB, true>;
    static const hipError_t attr = hipFuncSetAttribute((const void *)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, CF::LDS_BYTES);
    if (attr != hipSuccess) return hip_fail(attr, "hipFuncSetAttribute");
    timing_begin(s);
    hipLaunchKernelGGL(kern, dim3((unsigned)ntiles), dim3(CF::NT), CF::LDS_BYTES, s, 0, 0, 0,
                       (const typename FMT::E *)nullptr, 0L, 0, (const typename FMT::E *)nullptr, 0L, 0, 0.0f, 0.0f,
                       (float *)nullptr, 0L, 0, 0, (const unsigned *)nullptr, (const unsigned *)nullptr, Epilogue(),
                       (const float *)nullptr, 0L, (const float *)nullptr, 0L, 0, 0, (float *)nullptr, probs, tiles);
    timing_end(s);
    e = hipGetLastError();
    return e == hipSuccess ? UGEMM_OK : hip_fail(e, "grouped split-form core");
}

// Grouped-only variants (kNumVariants + i): base variant split_b_base(np, i)
// with B split in the core -- the 4-wave tiles with 128 B rows (each thread
// stages two rows of a row-contiguous B): 128 x 128, and 256 x 128; then
// the 8-wave streamed 128 x 128 (one row per thread).
constexpr int kNumSplitB = 3;
constexpr int split_b_base(int np, int i) { return i == 0 ? 1 : i == 2 ? 7 : (np == 3 ? 0 : 2); }

template <int NP, class FMT = FmtBf16>
int grouped_np(int variant, int b_kcont, const PrepJob *jobs, const int *block_job, int prep_blocks,
               const GroupedSplitProblem *probs, const GroupedSplitTile *tiles, int ntiles, hipStream_t s,
               const GroupedScales *sc) {
    using T = Table<NP, FMT>;
#define UGEMM_SPLIT_B(CFG)                                                                                    \
    (b_kcont ? grouped_core<CFG, FUSE_KCONT>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc)           \
             : grouped_core<CFG, FUSE_RCONT>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc))
    static_assert(split_b_base(NP, 0) == 1 && split_b_base(NP, 1) == (NP == 3 ? 0 : 2) && split_b_base(NP, 2) == 7,
                  "split-B table");
    switch (variant) {
        case kNumVariants + 0: return UGEMM_SPLIT_B(typename T::V1);
        case kNumVariants + 1:
            if constexpr (NP == 3) return UGEMM_SPLIT_B(typename T::V0);
            else return UGEMM_SPLIT_B(typename T::V2);
        case kNumVariants + 2: return UGEMM_SPLIT_B(typename T::V7);
        default: break;
    }
#undef UGEMM_SPLIT_B
    switch (variant) {
        case 0: return grouped_core<typename T::V0>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 1: return grouped_core<typename T::V1>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 2: return grouped_core<typename T::V2>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 3: return grouped_core<typename T::V3>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 4: return grouped_core<typename T::V4>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 5: return grouped_core<typename T::V5>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 6: return grouped_core<typename T::V6>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case 7: return grouped_core<typename T::V7>(jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        default: return fail(UGEMM_ERR_ARG, "grouped split form: no variant %d", variant);
    }
}

template <int NP, class FMT = FmtBf16>
void tile_of(int variant, int *bm, int *bn) {
    using T = Table<NP, FMT>;
    switch (variant) {
        case 0: *bm = T::V0::BM; *bn = T::V0::BN; break;
        case 1: *bm = T::V1::BM; *bn = T::V1::BN; break;
        case 2: *bm = T::V2::BM; *bn = T::V2::BN; break;
        case 3: *bm = T::V3::BM; *bn = T::V3::BN; break;
        case 4: *bm = T::V4::BM; *bn = T::V4::BN; break;
        case 5: *bm = T::V5::BM; *bn = T::V5::BN; break;
        case 6: *bm = T::V6::BM; *bn = T::V6::BN; break;
        default: *bm = T::V7::BM; *bn = T::V7::BN; break;
    }
}
}  // namespace

int mfma_grouped_variant_count(int mode) { return planes_of(mode) ? kNumVariants + kNumSplitB : 0; }

int mfma_grouped_splits_b(int mode, int variant) {
    return planes_of(mode) && variant >= kNumVariants && variant < kNumVariants + kNumSplitB ? 1 : 0;
}

const char *mfma_grouped_variant_name(int mode, int variant) {
    if (!planes_of(mode) || variant < 0 || variant >= kNumVariants + kNumSplitB) return nullptr;
    if (variant < kNumVariants) return mfma_variant_name(mode, variant);
    // Formatted once per (mode, variant); function-local static initialisation is thread-safe.
    static const std::string names[UGEMM_MODE_COUNT][kNumSplitB] = {
#define UGEMM_N(m, i) (std::string(mfma_variant_name(m, split_b_base(planes_of(m), i)) \
                                    ? mfma_variant_name(m, split_b_base(planes_of(m), i)) : "") + "_split_b")
        {UGEMM_N(0, 0), UGEMM_N(0, 1), UGEMM_N(0, 2)}, {UGEMM_N(1, 0), UGEMM_N(1, 1), UGEMM_N(1, 2)},
        {UGEMM_N(2, 0), UGEMM_N(2, 1), UGEMM_N(2, 2)}, {UGEMM_N(3, 0), UGEMM_N(3, 1), UGEMM_N(3, 2)},
        {UGEMM_N(4, 0), UGEMM_N(4, 1), UGEMM_N(4, 2)}, {UGEMM_N(5, 0), UGEMM_N(5, 1), UGEMM_N(5, 2)},
        {UGEMM_N(6, 0), UGEMM_N(6, 1), UGEMM_N(6, 2)}
#undef UGEMM_N
    };
    return names[mode][variant - kNumVariants].c_str();
}

int mfma_grouped_tile(int mode, int variant, int *bm, int *bn) {
    if (variant >= kNumVariants && variant < kNumVariants + kNumSplitB)
        variant = split_b_base(planes_of(mode), variant - kNumVariants);
    if (variant < 0 || variant >= kNumVariants) return fail(UGEMM_ERR_ARG, "grouped split form: no variant %d", variant);
    switch (mode) {
        case UGEMM_MODE_BF16X1: tile_of<1>(variant, bm, bn); return UGEMM_OK;
        case UGEMM_MODE_BF16X3: tile_of<2>(variant, bm, bn); return UGEMM_OK;
        case UGEMM_MODE_BF16X6: tile_of<3>(variant, bm, bn); return UGEMM_OK;
        case UGEMM_MODE_FP16X3: tile_of<2, FmtF16>(variant, bm, bn); return UGEMM_OK;
        default: return fail(UGEMM_ERR_UNSUPPORTED, "grouped: mode %d not provided", mode);
    }
}

int launch_mfma_grouped(int mode, int variant, int b_kcont, const PrepJob *jobs, const int *block_job,
                        int prep_blocks,
                        const GroupedSplitProblem *probs, const GroupedSplitTile *tiles, int ntiles, hipStream_t s,
                        const GroupedScales *sc) {
    if (ntiles == 0) return UGEMM_OK;
    switch (mode) {
        case UGEMM_MODE_BF16X1:
            return grouped_np<1>(variant, b_kcont, jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case UGEMM_MODE_BF16X3:
            return grouped_np<2>(variant, b_kcont, jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case UGEMM_MODE_BF16X6:
            return grouped_np<3>(variant, b_kcont, jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        case UGEMM_MODE_FP16X3:
            if (!sc) return fail(UGEMM_ERR_ARG, "grouped FP16X3: no row-scale jobs");
            return grouped_np<2, FmtF16>(variant, b_kcont, jobs, block_job, prep_blocks, probs, tiles, ntiles, s, sc);
        default: return fail(UGEMM_ERR_UNSUPPORTED, "grouped: mode %d not provided", mode);
    }
}

int launch_mfma_conv(const Gemm<float> &g, const ConvDesc &cd, int mode, int variant, hipStream_t s) {
    // No operand is split in the core here (the im2col operand is gathered
    // into planes), so the picker's fusing variant gives way to the
    // plane-streaming one.
    Gemm<float> gs = g;
    const int v = variant >= 0 ? variant : mfma_pick_variant(g, mode, false, &gs.splits);
    switch (mode) {
        case UGEMM_MODE_BF16X1: return launch_np_conv<1>(gs, cd, v, s);
        case UGEMM_MODE_BF16X3: return launch_np_conv<2>(gs, cd, v, s);
        case UGEMM_MODE_BF16X6: return launch_np_conv<3>(gs, cd, v, s);
        case UGEMM_MODE_FP16X3: return launch_np_conv<2, FmtF16>(gs, cd, v, s);
        default: return fail(UGEMM_ERR_UNSUPPORTED, "conv: mode %d is not provided", mode);
    }
}

int launch_mfma(const Gemm<float> &g, int mode, int variant, hipStream_t s) {
    // Variant 3 with the automatic split count: small grids in one launch.
    if (variant == 3 && g.splits == 0)
        if (const int tile = split_small_tile(g, mode)) return launch_split_small(g, mode, tile, s);
    switch (mode) {
        case UGEMM_MODE_BF16X1: return launch_np<1>(g, variant, s);
        case UGEMM_MODE_BF16X3: return launch_np<2>(g, variant, s);
        case UGEMM_MODE_BF16X6: return launch_np<3>(g, variant, s);
        case UGEMM_MODE_FP16X3: return launch_np<2, FmtF16>(g, variant, s);
        default: return fail(UGEMM_ERR_UNSUPPORTED, "mode %d is not a split form", mode);
    }
}

}  // namespace ugemm
