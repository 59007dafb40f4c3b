// fp32 GEMM of many rows on the bf16 matrix instruction (v_mfma_f32_16x16x32_bf16), with no bit of an operand left out:
//
//     C[M, N] = X[M, K] . W[N, K]^T        K % 32 == 0
//
// An fp32 value is the exact sum of three bf16 terms, its 24 bits in groups of eight.  Where W's values are bf16 ones (weights of a
// 16-bit checkpoint, widened), X . W is the sum of three products of bf16 operands, each of which the instruction forms exactly and
// adds in fp32: sixteen times the fp32 instruction's rate, for three times the products.  W stays 32 bits wide in memory and is
// looked at as it is read.  If a value has lower bits, is infinite (an infinity times a term of 0 is no number) or smaller than bf16's
// normal numbers (whose products the instruction forms with fewer bits), or if X has a value whose lowest bits would be finer than
// bf16's (below 2^-110), a flag is set and the fp32 instruction's form (gemm32.hip), which is launched behind and otherwise only adds
// slices, makes the whole result.  A workgroup that sees it in its first K-tile or its rows of X stops there, others when their next
// chain of 16 K-tiles ends.  What that costs, us, all in turn with rotating weights: 903 x 28672 x 4096 on the fp32 instruction 1603, by way of
// here with 24 bits in all of W 1577, in half of its rows 1598 (500 more where nobody asks the others), in half of its columns 1669, in its
// last value alone 2078; 160 x 6144 x 4096 75, 86, 101, 109, 115.  Each timed by itself the instruction takes 1536 at the former, and 24
// bits in all of W 1577.  What a model has loaded carries the answer and does not come here (ops/hip.py gemm32).
//
// Relative error (2-norm, random operands, K 4096 - 22528, chains of 16 K-tiles on both): 2.4e-7, the fp32 instruction 4.1e-7, as one
// sum takes the products of 32 columns and not of four.
//
// What bounds it: the arrival of the tiles, and the card's power.  A workgroup of four waves has up to 160 rows x 256 columns of
// outputs, one wave a SIMD with 80 x 128; larger ones do not fit in the registers beside the sums of finished chains.  A K-tile of 32 is
// 1920 cycles of products, 120 KiB of LDS reads and 62 KiB of requests, and takes 1.6 - 1.7 us (1.2 PFLOP/s in bf16, 0.9 us with the
// requests left out, 1.7 PFLOP/s at the clock that the power then allows).
//   * X's terms are made by a launch ahead (10 bytes a value), in the order that fragments are read in: 1 KiB pieces of
//     consecutive lanes, by LDS-DMA and by ds_read_b128 alike.
//   * W arrives by LDS-DMA too, 8 rows x 128 bytes an instruction; loaded by the lanes that use it (16 rows x 64 bytes) it took
//     three times as many cache accesses and as long (20608 columns, 300 rows: 181 us, 165 here).
//   * every product has an instruction or three of other work behind it: it keeps the matrix core busy for 16 cycles and the
//     wave for four.
//   * what is looked at in W takes a fifth of the instructions beside the products: each of the two waves that have the same columns
//     looks at half of them.  With the smallest value of all columns looked for in both, 903 x 4096 x 14336 took 8 % longer.
// us, fp32 instruction -> this: 903 x 28672 x 4096 1518 -> 564, 903 x 4096 x 14336 787 -> 315, 300 x 20608 x 4096 421 -> 165, 160 x
// 28672 x 4096 291 -> 151 (where W's arrival is all).  Which rows and shapes: ops/hip.py gemm32_terms.
#include "gemm32.h"

#include <type_traits>

namespace {
constexpr int BLOCK = 3072;             // bytes of a K-tile of 32 of 16 rows of X: [term][lane][16]
constexpr int WI = TN * 128, WS = 3;    // bytes of W's K-tile, and how many are in LDS; behind them X's
constexpr int x_slots(int nb) { return nb <= 3 ? 3 : 2; }
constexpr int LDS_BYTES = WS * WI + 2 * 2 * MAX_NB * BLOCK;
constexpr int TAIL = 512 + 3 * 1024;    // and behind these what is known of values that are not the sums of their terms
static_assert(LDS_BYTES + TAIL <= 160 * 1024 && x_slots(3) * 2 * 3 * BLOCK <= 2 * 2 * MAX_NB * BLOCK, "LDS");

typedef __attribute__((address_space(3))) void* lds_ptr;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}

__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302); }

// Values that terms hold short: a bf16 ends at 2^-133 and so do the lowest bits of x from 2^-110 up; below bf16's smallest normal
// number the products of w have fewer bits (x 2^20 times 2^-133: 7e-6 off).
constexpr uint32_t X_LEAST = (127 - 110) << 23;
constexpr uint32_t W_LEAST = 2 * 0x0080;  // of 2 d, d without its sign

// v - its first term; infinities leave none
__device__ __forceinline__ uint32_t below(uint32_t v) {
    const float top = __uint_as_float(v & 0xffff0000u);
    return (v & 0x7f800000u) == 0x7f800000u ? 0u : __float_as_uint(__uint_as_float(v) - top);
}
}  // namespace

// X's terms, laid out as the matrix instruction reads them: [M / 16][K / 32][term][lane][8], lane (r, g) holding row r, k 4 g .. and
// 16 + 4 g ..  Rows past M are zeros.  ``inexact`` is cleared; 16 bytes behind it, a byte for four pieces says whether X has a value
// there that is not the sum of its terms, and zeros up to a multiple of 16.
__global__ __launch_bounds__(256) void terms32_kernel(const float* __restrict__ x, int ldx, char* __restrict__ out, int M, int kb,
                                                      int pieces, int* inexact) {
    __shared__ uint32_t s_small[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = blockIdx.x * 4 + w;
    const int block = p / kb, kt = p - block * kb, m = block * 16 + (lane & 15);
    u32x4 v[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    if (m < M) {
        const u32x4* in = reinterpret_cast<const u32x4*>(x + (size_t)m * ldx + kt * 32) + (lane >> 4);
        v[0] = in[0];
        v[1] = in[4];
    }
    u32x4 t[3];
    bool small = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t a[2][3];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t u = v[i >> 1][2 * (i & 1) + j], r = below(u);
            small |= (u & 0x7fffffffu) - 1 < X_LEAST - 1;
            a[j][0] = (u & 0x7fffffffu) > 0x7f800000u ? u | 0x00400000u : u;  // a NaN whose bits are all low
            a[j][1] = r;
            a[j][2] = below(r);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) t[k][i] = high_halves(a[0][k], a[1][k]);
    }
    if (p < pieces) {
        u32x4* o = reinterpret_cast<u32x4*>(out + (size_t)p * BLOCK) + lane;
#pragma unroll
        for (int k = 0; k < 3; ++k) o[64 * k] = t[k];
    }
    const bool any = __ballot(small) != 0;
    if (lane == 0) s_small[w] = any;
    __syncthreads();
    char* flags = reinterpret_cast<char*>(inexact) + 16;
    if (threadIdx.x == 0) flags[blockIdx.x] = s_small[0] | s_small[1] | s_small[2] | s_small[3];
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) *inexact = 0;
        const int i = gridDim.x + threadIdx.x;
        if (threadIdx.x < 16 && i < (((int)gridDim.x + 15) & ~15)) flags[i] = 0;
    }
}

namespace {
// K-tiles [kt0, kt1) of 32 NB rows from 32 u0 on and columns n0 ..; wave (wr, wc) has half of the rows and 128 columns: acc[row
// block][column block ^ wr], so that the two waves that have the same columns each look at every other block of them, by the same
// code.  False: some value is not the sum of its terms, and the sums are not made.
template <int NB>
__device__ __forceinline__ bool terms_loop(const Gemm32Args& a, char* lds, int u0, int n0, int kt0, int kt1, f32x4 (&acc)[NB][8]) {
    constexpr int XI = 2 * NB * BLOCK, PX = (6 * NB + 3) / 4, XS = x_slots(NB);
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wr = w >> 1, wc = w & 1;
    const __amdgpu_buffer_rsrc_t rx = buffer(reinterpret_cast<const char*>(a.x) + (size_t)u0 * 2 * a.kb * BLOCK, 2 * NB * a.kb * BLOCK);
    const __amdgpu_buffer_rsrc_t rw = buffer(a.w + (size_t)n0 * a.ldw, min(a.N - n0, TN) * a.ldw * 4);
    // pieces of 1 KiB.  X: a term of a row block, every fourth one (behind the last that one again); W: 8 rows of this wave's 64,
    // position lane & 7 of row r taking chunk (lane & 7) ^ ((r >> 1) & 7); behind row N the last one again
    int vx[PX], dx[PX], vw[8];
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        const int p = min(w + 4 * i, 6 * NB - 1);
        vx[i] = (p / 3) * a.kb * BLOCK + p % 3 * 1024 + lane * 16;
        dx[i] = WS * WI + p * 1024;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = 64 * w + 8 * i + (lane >> 3);
        vw[i] = min(r, a.N - n0 - 1) * a.ldw * 4 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    auto stage_x = [&](int kt, int slot, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(lds + slot * XI + dx[i]), 16, vx[i], kt * BLOCK, 0, 0);
    };
    auto stage_w = [&](int kt, int slot, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(lds + slot * WI + (8 * w + i) * 1024), 16, vw[i], kt * 128, 0, 0);
    };
    const int wlo = (128 * wc + r16) * 128 + ((g ^ (r16 >> 1)) << 4), wl[2] = {wlo + wr * 2048, wlo - wr * 2048};
    const int xlo = WS * WI + wr * NB * BLOCK + lane * 16;
    auto read_w = [&](u32x4 (&q)[2], int slot, int i, int h) {
        q[h] = *reinterpret_cast<const u32x4*>(lds + slot * WI + (h ? wl[i & 1] ^ 64 : wl[i & 1]) + i * 2048);
    };
    auto read_x = [&](u32x4 (&x)[3], int slot, int b, int k) {
        x[k] = *reinterpret_cast<const u32x4*>(lds + slot * XI + xlo + b * BLOCK + k * 1024);
    };
    // First terms of a pair of W's values.  ``look``: and what they leave out: ``low`` gathers the bits below them, ``top`` the largest
    // size, and ``least`` the smallest one but zero, as 2 d - 1, in products of its own (written out, as the compiler would put a
    // wait on either side of such a minimum between written-out lines).
    uint32_t low = 0, least = 0xffffffff;
    float top = 0.f;
    auto first = [&](const u32x4 (&q)[2], u32x4& f, int i, bool look) {
        const uint32_t u = q[i >> 1][2 * (i & 1)], v = q[i >> 1][2 * (i & 1) + 1];
        uint32_t d = high_halves(u, v);
        if (look) {
            low |= u | v;
            top = fmaxf(fmaxf(top, fabsf(__uint_as_float(u))), fabsf(__uint_as_float(v)));
        }
        asm volatile("" : "+v"(d), "+v"(low), "+v"(top));  // here, and not where they are used
        f[i] = d;
    };
    auto smallest = [&](uint32_t d) {
        uint32_t e;
        asm volatile("v_pk_mad_u16 %1, %2, %3, %4\n\tv_pk_min_u16 %0, %0, %1"
                     : "+v"(least), "=&v"(e) : "v"(d), "s"(0x00020002), "v"(0xffffffff));
    };
    auto any = [&] {
        return __ballot((low & 0xffffu) != 0 || top == __builtin_inff() || min(least & 0xffffu, least >> 16) < W_LEAST - 1) != 0;
    };
    // The products are written out so that a block's sums stay in their registers (left to the compiler, they are copied from
    // one set to another every K-tile, and spilled).  The waits that it would put between them and other uses of these registers
    // stand at the ends of a K-tile.
    auto mfma = [](const u32x4& f, const u32x4& x, f32x4& c) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(f), "v"(x));
    };
    // this wave has read what it wanted, and all but its last N requests have arrived; and so in all waves
    auto meet = [](auto ahead) {
        constexpr int N = decltype(ahead)::value;
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const int last = kt1 - 1;
    // What X's split has found in this tile's rows (and, to whole 16 bytes, in some next to them) and whether another workgroup has
    // met something go to LDS ahead of the first K-tile, and are not waited for by themselves.
    int* heard = reinterpret_cast<int*>(lds + LDS_BYTES);        // word 0: the flag, as it was asked for last
    int* seen = heard + 64;
    const volatile int* words = heard + 128;
    const __amdgpu_buffer_rsrc_t rf = buffer(a.inexact, 4);
    auto ask = [&] { __builtin_amdgcn_raw_ptr_buffer_load_lds(rf, (lds_ptr)heard, 4, lane ? 4 : 0, 0, 0, 16); };
    const int flag0 = (2 * u0 * a.kb >> 2) & ~15, flags = ((((a.M + 31) >> 5) * 2 * a.kb + 3 >> 2) + 15 & ~15) - flag0;
    const int nwords = ((2 * (u0 + NB) * a.kb - 1 >> 2) - flag0 >> 2) + 1;
    const char* flag = reinterpret_cast<const char*>(a.inexact) + 16 + flag0;
    if (w == 3)
        ask();
    else if (256 * w < nwords)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(flag, flags), (lds_ptr)(heard + 128 + 256 * w), 16, w * 1024 + lane * 16, 0, 0, 0);
#pragma unroll
    for (int d = 0; d < WS; ++d) {
        if (d < 2)
#pragma unroll
            for (int i = 0; i < PX; ++i) stage_x(min(kt0 + d, last), d, i);
#pragma unroll
        for (int i = 0; i < 8; ++i) stage_w(min(kt0 + d, last), d, i);
    }
    int small = 0;
    for (int i = tid + 256 * 3; i < nwords; i += 256) small |= reinterpret_cast<const int*>(flag)[i];
    meet(std::integral_constant<int, 8>{});  // all but the third W
#pragma unroll
    for (int i = 0; i < 3; ++i) small |= words[min(tid + 256 * i, min(nwords, 768) - 1)];
    small |= *(volatile int*)heard;
    u32x4 wf[8], x0[3];
    f32x4 sum[NB][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        u32x4 q[2];
        read_w(q, 0, i, 0);
        read_w(q, 0, i, 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            first(q, wf[i], j, i % 2 == 0);
            if (i % 2 == 0) smallest(wf[i][j]);
        }
    }
    const bool odd = any() || __ballot(small != 0) != 0;
    if (lane == 0) seen[w] = odd;
#pragma unroll
    for (int k = 0; k < 3; ++k) read_x(x0, 0, 0, k);
    meet(std::integral_constant<int, 8>{});
    if (seen[0] | seen[1] | seen[2] | seen[3]) {  // most W that are not bf16 values show it here
        if (tid == 0) atomicOr(a.inexact, 1);
        __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
        return false;
    }
    if constexpr (XS == 3)
#pragma unroll
        for (int i = 0; i < PX; ++i) stage_x(min(kt0 + 2, last), 2, i);
    // requests behind X of the next K-tile and W of the one after it, at a K-tile's meeting
    constexpr int AHEAD = 8 + (XS == 3 ? PX : 0);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
            sum[b][i] = acc[b][i];
        }
    int sx = 0, sw = 1;  // slots of X(t) and W(t + 1)
    // A K-tile: 24 products a row block, and an instruction or three of other work behind each, which takes the time of four:
    // reads of X a row block ahead, reads and conversion of the next K-tile's W, behind the meeting requests.
    auto step = [&](int kt) {
        u32x4 x[2][3], wn[8], q[8][2];
#pragma unroll
        for (int k = 0; k < 3; ++k) x[0][k] = x0[k];
        const int pw = sw == 0 ? WS - 1 : sw - 1;  // where the W of this K-tile was
        int px = 0;
        asm volatile("s_nop 3");
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b == NB - 1) {
                meet(std::integral_constant<int, AHEAD>{});
                px = sx;
                sx = sx + 1 == XS ? 0 : sx + 1;
                sw = sw + 1 == WS ? 0 : sw + 1;
            }
#pragma unroll
            for (int m = 0; m < 24; ++m) {
                mfma(wf[m & 7], x[b & 1][2 - (m >> 3)], acc[b][m & 7]);
                if (m < 3) read_x(x[(b + 1) & 1], sx, b < NB - 1 ? b + 1 : 0, m);
                const int s = 24 * b + m;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int at = 3 * (NB - 1) * i;
                    if (s == at) read_w(q[i], sw, i, 0);
                    if (s == at + 1) read_w(q[i], sw, i, 1);
                    if (s >= at + 14 && s < at + 18) first(q[i], wn[i], s - at - 14, i % 2 == 0);
                    if (i % 2 == 0 && s >= at + 18 && s < at + 22) smallest(wn[i][s - at - 18]);
                    if (s == at + 2) stage_w(min(kt + WS, last), pw, i);
                }
                if (b == NB - 1 && m >= 4 && m < 4 + PX) stage_x(min(kt + XS, last), px, m - 4);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        asm volatile("s_nop 15\ns_nop 15");
#pragma unroll
        for (int i = 0; i < 8; ++i) wf[i] = wn[i];
#pragma unroll
        for (int k = 0; k < 3; ++k) x0[k] = x[NB & 1][k];
    };
    // Chains.  At the end of one the workgroup says what it has met and ends with it if another one has met something: what it stores
    // then is overwritten.  (Without a branch, and in the loop's bound: around one the compiler moves the sums about and spills.)
    for (int kt = kt0, stop = kt1; kt < stop;) {
        const int end = min(kt + LONG_RUN, kt1);
        for (; kt < end; ++kt) {
            // the flag arrives ahead of this K-tile's meeting and is read behind it; the next one is asked for LONG_RUN K-tiles later
            if (kt == end - 1 && end < kt1 && w == 0) ask();
            step(kt);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 8; i += 4) {
                asm volatile("s_nop 7" : "+a"(acc[b][i]), "+a"(acc[b][i + 1]), "+a"(acc[b][i + 2]), "+a"(acc[b][i + 3]));
#pragma unroll
                for (int j = i; j < i + 4; ++j) {
                    sum[b][j] += acc[b][j];
                    acc[b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                asm volatile("" : "+a"(acc[b][i]), "+a"(acc[b][i + 1]), "+a"(acc[b][i + 2]), "+a"(acc[b][i + 3]));
            }
        __builtin_amdgcn_raw_ptr_buffer_atomic_add_i32(1, rf, any() && lane == 0 ? 0 : 4, 0, 0);  // (at 4: nowhere)
        if (__builtin_amdgcn_readfirstlane(*(volatile int*)heard) && end < kt1) stop = kt;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[b][i] = sum[b][i];
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));  // nothing may arrive in LDS that another workgroup has by then
    return true;
}

template <int NB>
__device__ __forceinline__ void terms_tile(const Gemm32Args& a, char* lds, int u0, int n0, int kt0, int kt1, f32x4* part) {
    f32x4 acc[NB][8];
    if (!terms_loop<NB>(a, lds, u0, n0, kt0, kt1, acc)) return;
    const int tid = threadIdx.x;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (part) part[(b * 8 + i) * 256 + tid] = acc[b][i];
            else store_terms(a, u0, NB, n0, b, i, acc[b][i]);
        }
}
}  // namespace

__global__ __launch_bounds__(256, 1) void gemm32_terms_kernel(const Gemm32Args a) {
    __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES + TAIL];
    int p = blockIdx.x, slice = -1, kt0 = 0, kt1 = a.kb;
    if (p < a.whole) {
        p = xcd_position(p, a.whole);
    } else {
        const int rest = a.tiles_m * a.tiles_n - a.whole;
        p = xcd_position(p - a.whole, rest * a.splits);
        slice = p / rest;
        p += a.whole - slice * rest;
        kt0 = a.kb * slice / a.splits;
        kt1 = a.kb * (slice + 1) / a.splits;
    }
    int tm, tn, u0, nu;
    tile32(a, p, tm, tn);
    rows_of(a, (a.M + 31) >> 5, tm, tn, u0, nu);
    f32x4* part = slice < 0 ? nullptr : reinterpret_cast<f32x4*>(a.part + ((size_t)(p - a.whole) * a.splits + slice) * SLOT);
    switch (nu) {
        case 2: terms_tile<2>(a, lds, u0, tn * TN, kt0, kt1, part); break;
        case 3: terms_tile<3>(a, lds, u0, tn * TN, kt0, kt1, part); break;
        case 4: terms_tile<4>(a, lds, u0, tn * TN, kt0, kt1, part); break;
        default: terms_tile<5>(a, lds, u0, tn * TN, kt0, kt1, part); break;
    }
}

// *odd is set if one of n values is not a finite bf16 one, or is a subnormal one.  Bound by the reads: 28672 x 4096 in 88 us (5.3 TB/s).
__global__ __launch_bounds__(256) void bf16_values_kernel(const uint32_t* __restrict__ w, size_t n, int* odd) {
    const size_t step = (size_t)gridDim.x * 256, i0 = (size_t)blockIdx.x * 256 + threadIdx.x, n4 = (uintptr_t)w % 16 ? 0 : n / 4;
    bool any = false;
    auto look = [&](uint32_t u) {
        const uint32_t size = u & 0x7fffffffu;
        any |= (u & 0xffffu) != 0 || size >= 0x7f800000u || size - 1 < 0x00800000u - 1;
    };
    for (size_t i = i0; i < n4; i += 4 * step) {
        u32x4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = i + k * step < n4 ? reinterpret_cast<const u32x4*>(w)[i + k * step] : u32x4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) look(v[k][j]);
    }
    for (size_t i = 4 * n4 + i0; i < n; i += step) look(w[i]);
    if (__ballot(any) && (threadIdx.x & 63) == 0) atomicOr(odd, 1);
}

MRSUM_API int mrsum_bf16_values(const float* w, int rows, int cols, int* odd, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return 0;
    if (!w || !odd) return (int)hipErrorInvalidValue;
    const size_t n = (size_t)rows * cols;
    bf16_values_kernel<<<(int)std::min<size_t>(2048, (n + 4095) / 4096), 256, 0, s>>>(reinterpret_cast<const uint32_t*>(w), n, odd);
    return (int)hipGetLastError();
}

// terms: 2 ceil(M / 32) (K / 32) pieces of 3072 bytes, 16 bytes and a byte for four pieces, to a multiple of 16; on 16 bytes.  ``tiles_m``,
// ``whole``, ``splits``: row tiles of 2 to 5 32-row units, the rest from raster position ``whole`` on in slices of K through ``part``
// [tiles - whole][splits][40960], which the fp32 instruction's form with ``whole32``, ``splits32`` (mrsum_gemm32) uses too.
MRSUM_API int mrsum_gemm32_terms(const float* x, int ldx, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                                 int tiles_m, int whole, int splits, int whole32, int splits32, void* terms, float* part,
                                 hipStream_t s) {
    const int units = ceil_div(M, 32), kb = K / 32, tn = ceil_div(N, TN);
    if (M <= 32 || N <= 0 || K < 32 || K % 32 || ldx % 4 || ldw % 4 || (uintptr_t)x % 16 || (uintptr_t)w % 16 || !terms ||
        (uintptr_t)terms % 16 || tiles_m < 1 || units / tiles_m < 2 || ceil_div(units, tiles_m) > MAX_NB ||
        (size_t)TN * ldw * 4 >= (1u << 31) || (size_t)2 * MAX_NB * kb * BLOCK >= (1u << 31))
        return (int)hipErrorInvalidValue;
    const long long tiles = (long long)tiles_m * tn;
    if (splits < 1 || splits > kb || whole < 0 || whole > tiles || (splits > 1 && whole < tiles && !part) || splits32 < 1 ||
        tiles * std::max(splits, MAX_NB) >= (1ll << 31) || 2ll * units * kb >= (1ll << 31))
        return (int)hipErrorInvalidValue;
    const int pieces = 2 * units * kb;
    int* inexact = reinterpret_cast<int*>(static_cast<char*>(terms) + (size_t)pieces * BLOCK);
    Gemm32Args a{static_cast<const float*>(terms), w, c, 0, ldw, ldc, M, N, kb, tiles_m, tn, (int)tiles, 1, part, inexact};
    if (splits > 1) {
        a.whole = whole;
        a.splits = splits;
    }
    terms32_kernel<<<ceil_div(pieces, 4), 256, 0, s>>>(x, ldx, static_cast<char*>(terms), M, kb, pieces, inexact);
    gemm32_terms_kernel<<<a.whole + ((int)tiles - a.whole) * a.splits, 256, 0, s>>>(a);
    return gemm32_launch(x, ldx, w, ldw, c, ldc, M, N, K, whole32, splits32, part, &a, s);
}
