// What the fp32 GEMMs share: gemm32.hip (fp32 matrix instruction) and gemm32_terms.hip (bf16 instruction, three terms a value).
#pragma once
#include "common.h"

namespace {
// K-tiles whose products one chain of accumulations adds; the chains' sums are added in order, so that the error does not
// grow with K nor depend on how many slices a plan takes.  Relative error (2-norm, random operands), one chain -> this: K 4096
// 1.15e-6 -> 4.1e-7 (2.3e-7 of low tiles, whose slices may be four K-tiles long), K 22528 2.35e-6 -> 4.2e-7, for 1 % of the time
// (2 % at 20 - 64 rows).  Tall tiles of at most 16 K-tiles are one chain and run without the sums (gemm32_kernel<true>), which
// would be 5 - 9 % of so short a loop: 1200 x 16384 x 256 97.5 -> 89.2 us, 1500 x 8192 x 192 49.7 -> 46.0, 256 x 1024 x 512 17.4 -> 16.9.
constexpr int LONG_RUN = 16;
}  // namespace

struct Gemm32Args {
    const float* x;
    const float* w;
    float* c;
    int ldx, ldw, ldc, M, N, kb;  // kb: K-tiles
    int tiles_m, tiles_n;
    int whole, splits;  // raster positions from ``whole`` on run in ``splits`` slices of K
    float* part;        // [tiles - whole][splits][a tile's sums]
    int* inexact;       // terms: set where W has bits that its bf16 values lack
};

namespace {
// grouped raster: 8 tile rows of one tile column are neighbours.  A lone row tile needs no division, which are chains of some 40
// instructions ahead of a workgroup's first load: 20 x 8192 x 512 13.7 -> 13.1 us with this and the same in rows_of.
__device__ __forceinline__ void tile32(const Gemm32Args& a, int p, int& tm, int& tn) {
    if (a.tiles_m == 1) {
        tm = 0;
        tn = p;
        return;
    }
    const int gsz = 8 * a.tiles_n, g = p / gsz, first = 8 * g, gm = min(a.tiles_m - first, 8), within = p - g * gsz;
    tm = first + within % gm;
    tn = within / gm;
}

__device__ __forceinline__ void store_c(const Gemm32Args& a, int m, int n, const f32x4& v) {
    if (m >= a.M) return;
    float* o = a.c + (size_t)m * a.ldc + n;
    if (n + 4 <= a.N && a.ldc % 4 == 0 && (uintptr_t)a.c % 16 == 0) {
        *reinterpret_cast<f32x4*>(o) = v;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (n + j < a.N) o[j] = v[j];
    }
}

// Row tile tm of column tile tn: an even share of the ``blocks`` of rows, so that no tile is nearly empty beside full ones; which
// ones are a block taller changes from column to column, as two tall ones on a CU would set the time of all.
__device__ __forceinline__ void rows_of(const Gemm32Args& a, int blocks, int tm, int tn, int& b0, int& nb) {
    if (a.tiles_m == 1) {
        b0 = 0;
        nb = blocks;
        return;
    }
    const int turn = (tn + (tn >> 2) + (tn >> 4)) % a.tiles_m;
    b0 = (int)(((long long)blocks * tm + turn) / a.tiles_m);
    nb = (int)(((long long)blocks * (tm + 1) + turn) / a.tiles_m) - b0;
}

// tiles of the product in terms
constexpr int TN = 256;                 // columns
constexpr int MAX_NB = 5;               // 32-row units
constexpr int SLOT = MAX_NB * 32 * TN;  // scratch floats of a slice

// Outputs of (row block b, column block i ^ wr) of a tile of nb 32-row units: row lane & 15, columns 4 (lane >> 4) ..
__device__ __forceinline__ void store_terms(const Gemm32Args& a, int u0, int nb, int n0, int b, int i, const f32x4& v) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    store_c(a, 32 * u0 + 16 * (nb * (w >> 1) + b) + (lane & 15), n0 + 128 * (w & 1) + 16 * (i ^ (w >> 1)) + 4 * (lane >> 4), v);
}

// adds the slices of a split tile in terms: 2 x 16 rows of it, item = MAX_NB * (tile behind the whole ones) + unit
__device__ __forceinline__ void add_terms_slices(const Gemm32Args& a, int item) {
    const int tid = threadIdx.x, t = item / MAX_NB, b = item % MAX_NB;
    int tm, tn, u0, nu;
    tile32(a, a.whole + t, tm, tn);
    rows_of(a, (a.M + 31) >> 5, tm, tn, u0, nu);
    if (b >= nu) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * SLOT) + b * 8 * 256 + tid;
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = in[i * 256];
    for (int s = 1; s < a.splits; s += 2) {  // two slices in flight
        f32x4 q[2][8];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < 8; ++i) q[k][i] = in[(size_t)min(s + k, a.splits - 1) * (SLOT / 4) + i * 256];
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (s + k < a.splits)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] += q[k][i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) store_terms(a, u0, nu, tn * TN, b, i, v[i]);
}
}  // namespace

// the fp32 instruction's form; arguments as checked by mrsum_gemm32.  With ``terms``, a product in terms that is launched ahead: if its
// flag has been set the whole result, else what is left of that product
int gemm32_launch(const float* x, int ldx, const float* w, int ldw, float* c, int ldc, int M, int N, int K, int whole, int splits,
                  float* part, const Gemm32Args* terms, hipStream_t s);
