// Device-side helpers shared by the GEMM kernel families.
#pragma once

#include <hip/hip_runtime.h>
#include <utility>

namespace ugemm {

// static_for<N>(f): f(std::integral_constant<int, i>{}) for i = 0 .. N-1,
// unrolled at compile time (indices usable in if constexpr and templates).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Maps a launch's linear block id to a (tile_m, tile_n) pair of C tiles.
// 1) XCD de-interleave: hardware hands consecutive block ids round-robin to
//    the 8 XCDs of gfx950; renumber so that each XCD (one L2) owns a
//    contiguous range of tile ids.
// 2) Grouped order: GROUP_M tile-rows are walked column by column so that the
//    blocks resident at one time share A row-panels and B column-panels.
// The mapping is a bijection of [0, tiles_m * tiles_n).
__device__ __forceinline__ void tile_coords(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int total = tiles_m * tiles_n;
    int pid = bid;
    if ((total & 7) == 0) pid = (bid & 7) * (total >> 3) + (bid >> 3);
    constexpr int GROUP_M = 8;
    const int per_group = GROUP_M * tiles_n;
    const int group = pid / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = pid - group * per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// A 16-byte vector that needs only its element's alignment: a gfx950 global
// load or store of 16 bytes takes any 4-byte address, so operands with odd
// leading dimensions or offset bases move in the same 16-byte accesses as
// aligned ones.
template <typename T>
struct Vec16 {
    static constexpr int W = 16 / (int)sizeof(T);
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};
typedef Vec16<float>::type f32x4u;
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Loads one operand tile (a C_EXT x S_EXT block: C_EXT elements along the
// operand's contiguous dimension, S_EXT along its strided dimension) from
// global memory into registers, in chunks of 16 bytes (VEC elements).
//
// Edge tiles load without branches as well: a chunk that crosses the end of
// its row is loaded from the row's last VEC elements, a line past the last
// one from the last; mask(), called when the values are needed, shifts the
// cut chunks down and puts zeros in the place of what lies outside.  (Scalar
// loads under divergent branches, which this replaces for unaligned operands
// and cut chunks, ran an odd 4160 x 1152 x 1477 FP32 product at 30 TF/s; the
// masking next to the loads would make every step wait for its prefetch.)
template <typename T, int C_EXT, int S_EXT, int NT>
struct TileRegs {
    typedef typename Vec16<T>::type V;
    static constexpr int VEC = Vec16<T>::W;
    static constexpr int CHUNKS_C = C_EXT / VEC;
    static constexpr int NCHUNK = (C_EXT * S_EXT / VEC) / NT;
    static_assert((C_EXT * S_EXT / VEC) % NT == 0, "tile must split evenly over threads");
    V v[NCHUNK];

    // base points at the tile origin; element (c, s) is base[s * ld + c].
    __device__ __forceinline__ void load(const T *__restrict__ base, long ld, int t) {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
            const int f = t + i * NT;
            v[i] = *reinterpret_cast<const V *>(base + (long)(f / CHUNKS_C) * ld + (f % CHUNKS_C) * VEC);
        }
    }

    // cmax / smax: elements of a row, and lines, from the origin on (> 0).
    // wide: the operand's rows hold at least VEC elements (those before the
    // origin included); narrower ones are read element by element.
    __device__ __forceinline__ void load_edge(const T *__restrict__ base, long ld, int t, int cmax, int smax,
                                              bool wide) {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
            const int f = t + i * NT;
            const int c = (f % CHUNKS_C) * VEC;
            const int s = f / CHUNKS_C;
            const T *line = base + (long)min(s, smax - 1) * ld;
            if (wide) {
                v[i] = *reinterpret_cast<const V *>(line + min(c, cmax - VEC));
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[i][j] = line[min(c + j, cmax - 1)];
            }
        }
    }
    // After load_edge with the same arguments, before store.
    __device__ __forceinline__ void mask(int t, int cmax, int smax, bool wide) {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
            const int f = t + i * NT;
            const int c = (f % CHUNKS_C) * VEC;
            const int over = wide ? c + VEC - cmax : 0;   // > 0: elements of the chunk past the row's end
            V x = v[i];
            if constexpr (VEC == 4) {
                x = (over > 0 && (over & 1)) ? V{x[1], x[2], x[3], x[3]} : x;
                x = (over > 0 && (over & 2)) ? V{x[2], x[3], x[3], x[3]} : x;
            } else {
                x = (over > 0 && (over & 1)) ? V{x[1], x[1]} : x;
            }
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[i][j] = (f / CHUNKS_C < smax && c + j < cmax) ? x[j] : T(0);
        }
    }

    // Writes the registers into an LDS array L[k][x] of row length LD.
    // DIRECT: the contiguous dimension is x (the LDS fast index);
    // otherwise it is k and the chunk is written down a column.
    template <bool DIRECT, int LD>
    __device__ __forceinline__ void store(T *L, int t) const {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
            const int f = t + i * NT;
            const int c = (f % CHUNKS_C) * VEC;
            const int s = f / CHUNKS_C;
            if constexpr (DIRECT) {
                typedef T A16 __attribute__((ext_vector_type(VEC)));
                *reinterpret_cast<A16 *>(&L[s * LD + c]) = v[i];
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j) L[(c + j) * LD + s] = v[i][j];
            }
        }
    }
};

}  // namespace ugemm
