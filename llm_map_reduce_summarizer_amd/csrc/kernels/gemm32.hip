// fp32 GEMM on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32, no reduced-precision mode):
//
//     C[M, N] = X[M, K] . W[N, K]^T        K % 32 == 0
//
// A tile of up to 128 rows x 128 columns per 256-thread workgroup, two workgroups per CU; wave w owns all rows x columns
// [32 w, 32 w + 32), so that the four SIMDs have the same work at any number of 16-row blocks (in quarters of 64 x 64 a tile
// of 22 rows took as long as a full one: two of the SIMDs did its work).  The rows are dealt to the row tiles evenly.
// What bounds it is the matrix cores: a K-tile of 32 (128 bytes a row) is 128 instructions of 32 cycles a wave, 1.7 us, for 20
// LDS reads.  Images arrive by LDS-DMA, chunk c of row r at c ^ ((r >> 1) & 7) (conflict-free b128 fragment reads); the one
// wait and barrier of a K-tile stands in its middle, with the second half's fragments in registers, and the next
// K-tile's first ones are read behind the second half's products: both workgroups of a CU, which run in step, would else stop
// for their reads together (128 x 128 tiles, 480 -> 500 us with the reads ahead of the products they feed).
// us, four quarters, two barriers and one chain of sums -> this: 903 x 28672 x 4096 1653 -> 1530 (139 TFLOP/s of 155), 300 x
// 28672 x 4096 668 -> 567, 150 x 18560 x 4096 306 -> 199, 70 x 4096 x 8192 74 -> 55, 508 x 28672 x 4096 833 -> 844.  A workgroup
// costs 1 us more than there, which short calls of full tiles see: 128 x 2048 x 768 17.7 -> 18.3, 64 x 8192 x 384 13.3 -> 14.5.
// Tiles that would leave CUs idle run in slices of K (ops/hip.py _gemm32_plan), whose fp32 sums a second launch adds in slice
// order.  Short K runs in 64 x 64 tiles.
#include "gemm32.h"

#include <type_traits>

namespace {
constexpr int T32 = 128, STAGE = T32 * 128;  // bytes of W's K-tile
constexpr int LDS_BYTES = 80 * 1024;         // two workgroups on a CU
template <int NB>
constexpr int RUN = NB > 4 ? LONG_RUN : 4;

enum { PLAIN, PAST_CACHES };  // PAST_CACHES: W goes past the caches (gemm32_launch)
}  // namespace

// K-tiles [kt0, kt1) of a tile of NB row blocks; acc[row block][column block].  ONE: there are at most LONG_RUN of them
template <int NB, bool ONE, int FORM>
__device__ __forceinline__ void k_loop(const Gemm32Args& a, char* lds, int m0, int n0, int kt0, int kt1, f32x4 (&acc)[8][2]) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    constexpr int XB = NB * 2048, IMAGE = XB + STAGE, XI = (NB + 1) / 2;  // a K-tile of X; of both; pieces of X a wave
    constexpr int D = LDS_BYTES / IMAGE < 4 ? LDS_BYTES / IMAGE : 4;
    static_assert(D >= 2 && (D - 1) * (4 + XI) < 64, "K-tiles in flight");
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xrows = min(a.M - m0, 16 * NB), wrows = min(a.N - n0, T32);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + (size_t)m0 * a.ldx), (short)0, xrows * a.ldx * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.w + (size_t)n0 * a.ldw), (short)0, wrows * a.ldw * 4, 0x00020000);
    // staging: 8 rows per instruction, wave w rows 32 w .. 32 w + 31 of W and every fourth piece of X (behind the last one
    // that one again, so that all waves count alike); rows past M / N are dropped by the descriptor (their LDS rows feed
    // sums that are not stored)
    int vw[4], vx[XI], dx[XI];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 32 * w + 8 * i + (lane >> 3);
        vw[i] = r * a.ldw * 4 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int p = min(w + 4 * i, 2 * NB - 1), r = 8 * p + (lane >> 3);
        vx[i] = r * a.ldx * 4 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
        dx[i] = STAGE + p * 1024;
    }
    constexpr int NT = FORM == PAST_CACHES ? 2 : 0;  // nontemporal
    auto stage = [&](int kt, int buf) {
        char* dst = lds + buf * IMAGE;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(dst + (4 * w + i) * 1024), 16, vw[i], kt * 128, 0, NT);
#pragma unroll
        for (int i = 0; i < XI; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(dst + dx[i]), 16, vx[i], kt * 128, 0, 0);
    };
    int lo[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) lo[r] = (lane & 15) * 128 + (((4 * r + (lane >> 4)) ^ ((lane >> 1) & 7)) << 4);
    f32x4 xf[2][NB], wf[2][2];  // fragments of the two halves of a K-tile
    auto read = [&](int r, int buf) {
        const char* ws = lds + buf * IMAGE + w * 4096;
        const char* xs = lds + buf * IMAGE + STAGE;
#pragma unroll
        for (int i = 0; i < 2; ++i) wf[r][i] = *reinterpret_cast<const f32x4*>(ws + i * 2048 + lo[r]);
#pragma unroll
        for (int b = 0; b < NB; ++b) xf[r][b] = *reinterpret_cast<const f32x4*>(xs + b * 2048 + lo[r]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](int r) {
#pragma unroll
        for (int b = 0; b < NB; b += 2)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = b; q < b + 2 && q < NB; ++q)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        acc[q][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[r][i][j], xf[r][q][j], acc[q][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int PER = 4 + XI;  // requests of a wave for a K-tile
    // this wave's fragments are in registers and its pieces of the oldest K-tile but ``ahead`` have arrived, and so in all
    auto meet = [](auto ahead) {
        constexpr int N = decltype(ahead)::value * PER;
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int d = 0; d < D; ++d) stage(min(kt0 + d, kt1 - 1), d);
    meet(std::integral_constant<int, D - 1>{});
    read(0, 0);
    auto chain = [&](int& kt, int end, int& buf) {
        for (; kt < end; ++kt) {
            read(1, buf);
            products(0);
            meet(std::integral_constant<int, D - 2>{});
            stage(min(kt + D, kt1 - 1), buf);  // past the end the last one again, which nothing reads
            buf = buf + 1 == D ? 0 : buf + 1;
            read(0, buf);
            products(1);
        }
    };
    int kt = kt0, buf = 0;
    if constexpr (ONE && RUN<NB> == LONG_RUN) {
        chain(kt, kt1, buf);
    } else {
        f32x4 sum[NB][2];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i) sum[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        while (kt < kt1) {
            chain(kt, min(kt + RUN<NB>, kt1), buf);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    sum[b][i] += acc[b][i];
                    acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[b][i] = sum[b][i];
    }
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));  // nothing may arrive in LDS that another workgroup has by then
}

namespace {
template <bool ONE, int FORM>
__device__ __forceinline__ void tile_or_slice(const Gemm32Args& a, char* lds) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // an XCD's workgroups take neighbouring tiles: they share W's panels, and each XCD has taller and lower tiles alike
    int p = blockIdx.x, slice = -1, kt0 = 0, kt1 = a.kb;
    if (p < a.whole) {
        p = xcd_position(p, a.whole);
    } else {
        const int rest = a.tiles_m * a.tiles_n - a.whole;
        // short K: the slices of a tile on different XCDs.  us, one range of K to an XCD -> this: 508 x 2048 x 768 28.7 -> 25.4, 256 x
        // 4096 x 768 28.6 -> 25.9, 903 x 2048 x 512 31.9 -> 28.1; at K 1536 it costs up to 7 % (400 x 4096: 52 -> 56)
        p = a.kb > 32 ? xcd_position(p - a.whole, rest * a.splits) : p - a.whole;
        slice = p / rest;
        p += a.whole - slice * rest;
        kt0 = a.kb * slice / a.splits;
        kt1 = a.kb * (slice + 1) / a.splits;
    }
    int tm, tn, b0, nb;
    tile32(a, p, tm, tn);
    rows_of(a, (a.M + 15) >> 4, tm, tn, b0, nb);
    const int m0 = b0 * 16, n0 = tn * T32;
    f32x4 acc[8][2];
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#define LOOP(NB_) k_loop<NB_, ONE, FORM>(a, lds, m0, n0, kt0, kt1, acc)
    if constexpr (FORM == PAST_CACHES) {
        switch (nb) {
            case 1: LOOP(1); break;
            case 2: LOOP(2); break;
            default: LOOP(3); break;
        }
    } else {
        switch (nb) {
            case 1: LOOP(1); break;
            case 2: LOOP(2); break;
            case 3: LOOP(3); break;
            case 4: LOOP(4); break;
            case 5: LOOP(5); break;
            case 6: LOOP(6); break;
            case 7: LOOP(7); break;
            default: LOOP(8); break;
        }
    }
#undef LOOP
    if (slice >= 0) {
        f32x4* out = reinterpret_cast<f32x4*>(a.part + ((size_t)(p - a.whole) * a.splits + slice) * (T32 * T32)) + tid;
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (b < nb)
#pragma unroll
                for (int i = 0; i < 2; ++i) out[(b * 2 + i) * 256] = acc[b][i];
        return;
    }
#pragma unroll
    for (int b = 0; b < 8; ++b)
        if (b < nb)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                store_c(a, m0 + 16 * b + (lane & 15), n0 + 32 * w + 16 * i + 4 * (lane >> 4), acc[b][i]);
}

}  // namespace

template <bool ONE, int FORM>
__global__ __launch_bounds__(256, 2) void gemm32_kernel(const Gemm32Args a) {
    __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
    tile_or_slice<ONE, FORM>(a, lds);
}

// Behind a product in terms: adds what slices that has, or makes the whole result if it has met a value that terms hold short.
// (Forms of their own: the test of a pointer that is not there cost every other call 0.2 us, 16 x 768 x 768 8.1 -> 7.9.)  A launch that
// only looks at the flag takes 4 us.  us, the slices added by one of their own ahead -> here: 700 x 2048 x 2048 44 -> 39, 160 x 6144 x
// 4096 56 -> 51, 300 x 4096 x 14336 126 -> 117, 903 x 4096 x 8192 200 -> 197; of 24 bits, which no longer adds them: 86 -> 75, 96 -> 85,
// 347 -> 324, 522 -> 503.  (Without the launch below too, the last slice of a tile to arrive adding them all, 160 x 6144 took 50 and of
// 24 bits 142: each workgroup's slice has to leave its L2.)
template <bool ONE>
__global__ __launch_bounds__(256, 2) void gemm32_behind_kernel(const Gemm32Args a, const Gemm32Args terms) {
    __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
    if (!*terms.inexact) {
        if ((int)blockIdx.x < (terms.tiles_m * terms.tiles_n - terms.whole) * MAX_NB) add_terms_slices(terms, blockIdx.x);
        return;
    }
    if ((int)blockIdx.x < a.whole + (a.tiles_m * a.tiles_n - a.whole) * a.splits) tile_or_slice<ONE, PLAIN>(a, lds);
}

// adds the slices of the split tiles; one workgroup per (tile, 2 x 16 rows)
template <bool GUARD>
__global__ __launch_bounds__(256) void gemm32_tail_kernel(const Gemm32Args a, const int* inexact) {
    if (GUARD && !*inexact) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, t = blockIdx.x >> 2, b = 2 * (blockIdx.x & 3);
    int tm, tn, b0, nb;
    tile32(a, a.whole + t, tm, tn);
    rows_of(a, (a.M + 15) >> 4, tm, tn, b0, nb);
    if (b >= nb) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * (T32 * T32)) + b * 2 * 256 + tid;
    f32x4 v[4];
    const int n = b + 1 < nb ? 4 : 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = in[min(i, n - 1) * 256];
    for (int s = 1; s < a.splits; s += 4) {  // four slices in flight
        f32x4 p[4][4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) p[k][i] = in[(size_t)min(s + k, a.splits - 1) * (T32 * T32 / 4) + min(i, n - 1) * 256];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (s + k < a.splits)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] += p[k][i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < n)
            store_c(a, 16 * (b0 + b + (i >> 1)) + (lane & 15), tn * T32 + 32 * w + 16 * (i & 1) + 4 * (lane >> 4), v[i]);
}

// Short K: 64 x 64 tiles, loads and products in turns, wave w rows [16 w, 16 w + 16).  A K-tile takes half the time that a
// lone workgroup of the larger tiles takes, and four times as many workgroups share a small product (700 x 8192 x 192: 31 us
// in 128 x 128 tiles, 26 here); from K 512 on the larger tiles' rate leads.  Which one: ops/hip.py gemm32_small.
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

int gemm32_launch(const float* x, int ldx, const float* w, int ldw, float* c, int ldc, int M, int N, int K, int whole, int splits,
                  float* part, const Gemm32Args* terms, hipStream_t s) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 32 || ldx % 4 || ldw % 4 || (uintptr_t)x % 16 || (uintptr_t)w % 16 || (size_t)T32 * ldx * 4 >= (1u << 31) ||
        (size_t)T32 * ldw * 4 >= (1u << 31))
        return (int)hipErrorInvalidValue;
    if (splits && K < 32) return (int)hipErrorInvalidValue;  // the tiles ask for their first K-tiles ahead
    if (splits == 0) {
        if (ceil_div(M, TS) > 65535) return (int)hipErrorInvalidValue;
        gemm32_small_kernel<<<dim3(ceil_div(N, TS), ceil_div(M, TS)), 256, 0, s>>>(x, ldx, w, ldw, c, ldc, M, N, K);
        return (int)hipGetLastError();
    }
    Gemm32Args a{x, w, c, ldx, ldw, ldc, M, N, K / 32, ceil_div(M, T32), ceil_div(N, T32), 0, 1, part, nullptr};
    const int tiles = a.tiles_m * a.tiles_n;
    if (splits > 1 && (whole < 0 || whole >= tiles || splits > a.kb || !part)) return (int)hipErrorInvalidValue;
    a.whole = splits > 1 ? whole : tiles;
    a.splits = splits > 1 ? splits : 1;
    const int rest = tiles - a.whole;
    // Up to 48 rows are one row of tiles, which read W once a call; W of more than the 256 MiB that the last cache holds is gone by
    // the next call and goes past the caches.  us through the caches -> past them, the same W again / another one each time, K 4096: 4
    // x 14336 (224 MiB) 38.2 -> 42.9 / 53.8 -> 49.6, 4 x 16384 (256 MiB) 47.6 -> 55.7 / 60.0 -> 56.4, 4 x 18432 59.7 -> 57.6 / 65.1 ->
    // 60.2, 4 x 20608 67.3 -> 60.5 / 69.7 -> 62.8; 4 x 4096 15.8 -> 17.2 / 18.4 -> 18.0; 4 x 128256 399 -> 369 (5.7 TB/s).
    const bool once = M <= 48 && (size_t)N * K * 4 > (256u << 20);
    const int mine = a.whole + rest * a.splits;
    const int grid = terms ? std::max(mine, (terms->tiles_m * terms->tiles_n - terms->whole) * MAX_NB) : mine;
#define FORMS(ONE)                                                          \
    if (terms) gemm32_behind_kernel<ONE><<<grid, 256, 0, s>>>(a, *terms); \
    else if (once) gemm32_kernel<ONE, PAST_CACHES><<<grid, 256, 0, s>>>(a);  \
    else gemm32_kernel<ONE, PLAIN><<<grid, 256, 0, s>>>(a)
    if (ceil_div(a.kb, a.whole ? 1 : a.splits) <= LONG_RUN) {
        FORMS(true);
    } else {
        FORMS(false);
    }
#undef FORMS
    if (!rest) return (int)hipGetLastError();
    if (terms) gemm32_tail_kernel<true><<<rest * 4, 256, 0, s>>>(a, terms->inexact);
    else gemm32_tail_kernel<false><<<rest * 4, 256, 0, s>>>(a, nullptr);
    return (int)hipGetLastError();
}

// x [M][ldx], w [N][ldw], c [M][ldc]; tiles from raster position ``whole`` on in ``splits`` slices of K through ``part``
// [tiles - whole][splits][16384] (splits 1: none, part unused); splits 0: 64 x 64 tiles
MRSUM_API int mrsum_gemm32(const float* x, int ldx, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                           int whole, int splits, float* part, hipStream_t s) {
    return gemm32_launch(x, ldx, w, ldw, c, ldc, M, N, K, whole, splits, part, nullptr, s);
}
