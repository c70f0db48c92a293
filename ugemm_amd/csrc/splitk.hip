// Split-K support shared by the FP32, split-form and FP64 kernels: the split
// count heuristic and the fixed-order reduction of the partial products.
#include <algorithm>
#include <cmath>

#include "internal.h"

namespace ugemm {
namespace {

// C[m, n] = alpha * sum_{z < S} ws[z][m, n] + beta * C[m, n] (C not read when
// beta == 0), then the epilogue; the slices are added in z order.
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce(int M, int N, int S, T alpha, const T *__restrict__ ws, T beta,
                                                     T *__restrict__ C, long ldc, Epilogue epi) {
    const long total = (long)M * N, slice = total;
    const bool has_epi = epi.active();
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        T acc = ws[i];
        for (int z = 1; z < S; ++z) acc += ws[z * slice + i];
        const int m = (int)(i / N), n = (int)(i - (long)m * N);
        T *cp = C + (long)m * ldc + n;
        T v = beta == T(0) ? alpha * acc : fma(alpha, acc, beta * *cp);
        if constexpr (sizeof(T) == 4) {
            if (has_epi) v = apply_epilogue(epi, v, m, n);
        }
        *cp = v;
    }
}

template <typename T>
int reduce(int M, int N, int S, T alpha, const T *ws, T beta, T *C, long ldc, const Epilogue &epi, hipStream_t s) {
    const long total = (long)M * N;
    const long blocks = std::max<long>(1, std::min<long>((total + 255) / 256, 16L * device_cu_count()));
    hipLaunchKernelGGL(splitk_reduce<T>, dim3((unsigned)blocks), dim3(256), 0, s, M, N, S, alpha, ws, beta, C, ldc,
                       epi);
    UGEMM_HIP_TRY(hipGetLastError());
    return UGEMM_OK;
}

}  // namespace

int split_count(int requested, long tiles, int K, int kalign, int *kc, int per_cu) {
    int S = requested;
    if (S <= 0) {
        // Auto: split only when the grid fills at most half of the wanted
        // per_cu blocks on every CU, enough to reach that, with at least
        // 512 K per split.
        const long want = (long)per_cu * device_cu_count();
        S = 1;
        if (tiles * 2 <= want) S = (int)std::min<long>({want / std::max<long>(1, tiles), (long)K / 512, 16L});
        S = std::max(S, 1);
    }
    int chunk = (K + S - 1) / S;
    chunk = (chunk + kalign - 1) / kalign * kalign;
    if (chunk <= 0) chunk = kalign;
    S = std::max(1, (K + chunk - 1) / chunk);   // every split has a non-empty K range
    *kc = chunk;
    return S;
}

// The estimate behind the choice, fitted to sweeps of split counts 1-32 and of
// the grouped kernel over 64..1600 square C and K 200..50176 (FP32, FP32-MFMA,
// FP64; it is within 15% of the best measured choice there): the CU with the
// most blocks sets the time; o blocks on a CU lose 0.3 / o of it to latency (a
// workgroup of four groups counts as four); a chunk pays 64 of K for its first
// loads and its epilogue; the partial sums cost 50 S / K of the products and a
// second launch 5 us.
// 1400x1024x4096 FP32-MFMA: 205 us with the two-blocks-a-CU rule, 137 with
// this; 1000x600x5000 FP32 143 and 106; 1024x1024x2048 FP64 95 and 82 (groups).
bool deal_k(long tiles, int K, double us_per_k1000, int grouped, size_t c_bytes, int *splits) {
    const double cus = (double)device_cu_count(), t1 = us_per_k1000 * K / 1000.0;
    const double groups = t1 * std::ceil(tiles / cus) * (1.0 + 0.3 / 4) + 3.0;
    double best = 0;
    *splits = 1;
    // At most 32 MiB of partial sums: half the scratch of the no-allocation entry.
    for (int S = 1; S <= 32 && (S == 1 || (K / S >= 256 && S * c_bytes <= (32u << 20))); ++S) {
        const double most = std::ceil(tiles * S / cus), o = std::min(most, 5.0);
        double t = t1 * most / S * (1.0 + 0.3 / o) * (1.0 + 64.0 * S / K);
        if (S > 1) t = t * (1.0 + 50.0 * S / K) + 5.0;
        if (S == 1 || t < best) {
            best = t;
            *splits = S;
        }
    }
    return tiles <= grouped * cus && groups <= best;
}

int cheapest_tile(const TileCost *c, int n, unsigned skip, int v, int M, int N) {
    const long cus = device_cu_count();
    auto tiles = [&](const TileCost &t) { return (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn); };
    auto us = [&](const TileCost &t) { return t.us * t.bm * t.bn * ((double)((tiles(t) + cus - 1) / cus) + t.lone); };
    double best = 0.95 * us(c[v]);
    for (int i = 0; i < n; ++i) {
        if (skip >> i & 1 || tiles(c[i]) <= cus) continue;   // at most one tile a CU: split counts decide
        if (const double t = us(c[i]); t < best) {
            best = t;
            v = i;
        }
    }
    return v;
}

int launch_splitk_reduce_f32(int M, int N, int splits, float alpha, const float *ws, float beta, float *C, long ldc,
                             const Epilogue &epi, hipStream_t s) {
    return reduce<float>(M, N, splits, alpha, ws, beta, C, ldc, epi, s);
}
int launch_splitk_reduce_f64(int M, int N, int splits, double alpha, const double *ws, double beta, double *C,
                             long ldc, hipStream_t s) {
    return reduce<double>(M, N, splits, alpha, ws, beta, C, ldc, Epilogue(), s);
}

}  // namespace ugemm
