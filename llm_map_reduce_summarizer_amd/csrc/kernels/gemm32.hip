// fp32 GEMM on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32, no reduced-precision mode):
//
//     C[M, N] = X[M, K] . W[N, K]^T        K % 32 == 0
//
// 128 x 128 output tile per 256-thread workgroup, two workgroups per CU; wave (wr, wc) owns 64 x 64 outputs as 4 x 4
// blocks, or for M <= 64 (LOW) wave w 64 x 32, so that all four SIMDs have work (64 x 28672 x 4096: 248 -> 145 us; a form
// of its own: a branch cost the others 9 %).  K-tiles of 32 (128 bytes a row) arrive by LDS-DMA in two buffers, chunk c of
// row r at c ^ ((r >> 1) & 7) (conflict-free b128 fragment reads); a fragment's four floats feed four instructions, so a
// K-tile is 16 LDS reads for 128 instructions of 32 cycles, and the matrix cores set the time (1.7 us a K-tile) once a CU
// has work.  16-row blocks past M are skipped.  903 x 28672 x 4096: 2310 (64 x 64 tiles, loads between barriers) -> 1650
// us, 129 TFLOP/s of 157 and 146 counting the rows that pad the last tile.  Tiles that would leave CUs idle run in slices
// of K (ops/hip.py gemm32_splits), whose fp32 sums a second launch adds in slice order.  Short K runs in 64 x 64 tiles.
#include "common.h"

#include <type_traits>

namespace {
constexpr int T32 = 128, STAGE = T32 * 128;  // bytes of one operand's K-tile

struct Gemm32Args {
    const float* x;
    const float* w;
    float* c;
    int ldx, ldw, ldc, M, N, kb;  // kb: K-tiles
    int tiles_m, tiles_n;
    int whole, splits;  // raster positions from ``whole`` on run in ``splits`` slices of K
    float* part;        // [tiles - whole][splits][128 * 128]
};

// grouped raster: 8 tile rows of one tile column are neighbours
__device__ __forceinline__ void tile32(const Gemm32Args& a, int p, int& tm, int& tn) {
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
}  // namespace

template <bool LOW>
__global__ __launch_bounds__(256, 2) void gemm32_kernel(const Gemm32Args a) {
    __shared__ __attribute__((aligned(1024))) char lds[4 * STAGE];  // [buffer][x | w]
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wr = w >> 1, wc = w & 1;
    int p = blockIdx.x, slice = -1, kt0 = 0, kt1 = a.kb;
    if (p >= a.whole) {
        const int rest = a.tiles_m * a.tiles_n - a.whole;
        slice = (p - a.whole) / rest;
        p -= slice * rest;
        kt0 = a.kb * slice / a.splits;
        kt1 = a.kb * (slice + 1) / a.splits;
    }
    int tm, tn;
    tile32(a, p, tm, tn);
    const int m0 = tm * T32, n0 = tn * T32, xrows = min(a.M - m0, T32), wrows = min(a.N - n0, T32);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + (size_t)m0 * a.ldx), (short)0, xrows * a.ldx * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.w + (size_t)n0 * a.ldw), (short)0, wrows * a.ldw * 4, 0x00020000);
    // staging: wave w fills rows 32 w .. 32 w + 31 of both operands, 8 rows per instruction; rows past M / N are
    // dropped by the descriptor (their LDS rows feed sums that are not stored)
    const int row = 32 * w + (lane >> 3);
    const int ch0 = ((lane & 7) ^ ((lane >> 4) & 7)) << 4, ch1 = ((lane & 7) ^ ((4 + (lane >> 4)) & 7)) << 4;
    auto stage = [&](int kt, int buf) {
        char* dst = lds + buf * 2 * STAGE + w * 4096;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = i & 1 ? ch1 : ch0;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(dst + i * 1024), 16, (row + 8 * i) * a.ldx * 4 + ch,
                                                     kt * 128, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(dst + STAGE + i * 1024), 16,
                                                     (row + 8 * i) * a.ldw * 4 + ch, kt * 128, 0, 0);
        }
    };
    int lo[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) lo[r] = (lane & 15) * 128 + (((4 * r + (lane >> 4)) ^ ((lane >> 1) & 7)) << 4);
    constexpr int NC = LOW ? 2 : 4;
    f32x4 acc[4][NC];  // [row block][column block]
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < NC; ++i) acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int rbase = LOW ? 0 : 64 * wr, cbase = LOW ? 32 * w : 64 * wc;  // this wave's outputs
    const int nb = min(4, (xrows - rbase + 15) >> 4);                     // its row blocks (<= 0: none)
    auto compute = [&](int buf, auto all) {
        const char* xs = lds + buf * 2 * STAGE + rbase * 128;
        const char* ws = lds + buf * 2 * STAGE + STAGE + cbase * 128;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            f32x4 xf[4], wf[NC];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < NC) wf[i] = *reinterpret_cast<const f32x4*>(ws + i * 2048 + lo[r]);
                xf[i] = *reinterpret_cast<const f32x4*>(xs + i * 2048 + lo[r]);
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if (!decltype(all)::value && b >= nb) break;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < NC; ++i)
                        acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][j], xf[b][j], acc[b][i], 0, 0, 0);
            }
        }
    };
    auto bar = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    stage(kt0, 0);
    for (int kt = kt0, buf = 0; kt < kt1; ++kt, buf ^= 1) {
        if (kt + 1 < kt1) {
            stage(kt + 1, buf ^ 1);
            __builtin_amdgcn_s_waitcnt(8 | (7 << 4) | (15 << 8));  // vmcnt(8): all but the tile just asked for
        } else {
            __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
        }
        bar();
        if (nb == 4) compute(buf, std::true_type{});
        else if (nb > 0) compute(buf, std::false_type{});
        bar();
    }
    if (slice >= 0) {
        f32x4* out = reinterpret_cast<f32x4*>(a.part + ((size_t)(p - a.whole) * a.splits + slice) * (T32 * T32)) + tid;
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b < nb)
#pragma unroll
                for (int i = 0; i < NC; ++i) out[(b * 4 + i) * 256] = acc[b][i];
        return;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < NC; ++i)
            store_c(a, m0 + rbase + 16 * b + (lane & 15), n0 + cbase + 16 * i + 4 * (lane >> 4), acc[b][i]);
}

// adds the slices of the split tiles; one workgroup per (tile, 2 x 16 rows)
template <bool LOW>
__global__ __launch_bounds__(256) void gemm32_tail_kernel(const Gemm32Args a) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, t = blockIdx.x >> 2, b = blockIdx.x & 3;
    int tm, tn;
    tile32(a, a.whole + t, tm, tn);
    constexpr int NC = LOW ? 2 : 4;
    const int m = tm * T32 + (LOW ? 0 : 64 * (w >> 1)) + 16 * b, n = tn * T32 + (LOW ? 32 * w : 64 * (w & 1));
    if (m >= a.M) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * (T32 * T32)) + b * 4 * 256 + tid;
    f32x4 v[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) v[i] = in[i * 256];
    for (int s = 1; s < a.splits; ++s) {
        in += T32 * T32 / 4;
#pragma unroll
        for (int i = 0; i < NC; ++i) v[i] += in[i * 256];
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) store_c(a, m + (lane & 15), n + 16 * i + 4 * (lane >> 4), v[i]);
}

// Short K: 64 x 64 tiles, loads and products in turns, wave w rows [16 w, 16 w + 16).  A K-tile takes half the time that a
// lone workgroup of the larger tiles takes, and four times as many workgroups share a small product (256 x 4096 x 256: 22 us
// in 128 x 128 tiles, 12 here); from K 512 on the larger tiles' rate leads.  Which one: ops/hip.py gemm32_small.
constexpr int TS = 64, LDS32 = 32 + 4;  // tile, padded row of a K-tile

__global__ __launch_bounds__(256) void gemm32_small_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w,
                                                           int ldw, float* __restrict__ c, int ldc, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float sx[TS * LDS32];
    __shared__ __attribute__((aligned(16))) float sw[TS * LDS32];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int m0 = blockIdx.y * TS, n0 = blockIdx.x * TS;
    const int lr = tid >> 3, lc = (tid & 7) * 4;  // staging: rows lr and lr + 32, 4 columns
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int r16 = lane & 15, kq = lane >> 4;
    for (int k0 = 0; k0 < K; k0 += 32) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = lr + 32 * i;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
            if (m0 + r < M) a = *reinterpret_cast<const float4*>(x + (size_t)(m0 + r) * ldx + k0 + lc);
            if (n0 + r < N) b = *reinterpret_cast<const float4*>(w + (size_t)(n0 + r) * ldw + k0 + lc);
            *reinterpret_cast<float4*>(sx + r * LDS32 + lc) = a;
            *reinterpret_cast<float4*>(sw + r * LDS32 + lc) = b;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 32; k += 4) {
            const float a = sx[(16 * wv + r16) * LDS32 + k + kq];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, sw[(16 * i + r16) * LDS32 + k + kq], acc[i], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + 16 * i + r16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + 16 * wv + 4 * kq + j;
            if (m < M && n < N) c[(size_t)m * ldc + n] = acc[i][j];
        }
    }
}

// x [M][ldx], w [N][ldw], c [M][ldc]; tiles from raster position ``whole`` on in ``splits`` slices of K through ``part``
// [tiles - whole][splits][16384] (splits 1: none, part unused); splits 0: 64 x 64 tiles
MRSUM_API int mrsum_gemm32(const float* x, int ldx, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                           int whole, int splits, float* part, hipStream_t s) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 32 || ldx % 4 || ldw % 4 || (uintptr_t)x % 16 || (uintptr_t)w % 16 || (size_t)T32 * ldx * 4 >= (1u << 31) ||
        (size_t)T32 * ldw * 4 >= (1u << 31))
        return (int)hipErrorInvalidValue;
    if (splits == 0) {
        if (ceil_div(M, TS) > 65535) return (int)hipErrorInvalidValue;
        gemm32_small_kernel<<<dim3(ceil_div(N, TS), ceil_div(M, TS)), 256, 0, s>>>(x, ldx, w, ldw, c, ldc, M, N, K);
        return (int)hipGetLastError();
    }
    Gemm32Args a{x, w, c, ldx, ldw, ldc, M, N, K / 32, ceil_div(M, T32), ceil_div(N, T32), 0, 1, part};
    const int tiles = a.tiles_m * a.tiles_n;
    if (splits > 1 && (whole < 0 || whole >= tiles || splits > a.kb || !part)) return (int)hipErrorInvalidValue;
    a.whole = splits > 1 ? whole : tiles;
    a.splits = splits > 1 ? splits : 1;
    const int rest = tiles - a.whole;
    if (M <= 64) {
        gemm32_kernel<true><<<a.whole + rest * a.splits, 256, 0, s>>>(a);
        if (rest) gemm32_tail_kernel<true><<<rest * 4, 256, 0, s>>>(a);
    } else {
        gemm32_kernel<false><<<a.whole + rest * a.splits, 256, 0, s>>>(a);
        if (rest) gemm32_tail_kernel<false><<<rest * 4, 256, 0, s>>>(a);
    }
    return (int)hipGetLastError();
}
