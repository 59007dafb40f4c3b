// Chunked state-space scan of fp32 models on the fp32 matrix instruction (prompt portions): the form of ssm_chunk.hip,
// with every operand, weight and sum in fp32.  Chunks of 64 rows; with c_i the running sum of a dt over the chunk
// (log2 units), per head
//
//   M[i][j] = (C_i . B_j) 2^(c_i - c_j) dt_j  (j <= i)          y_i = sum_j M[i][j] x_j + 2^(c_i) (S C_i) + D x_i
//   S      <- 2^(c_last) S + sum_j 2^(c_last - c_j) dt_j x_j B_j^T
//
// dt and c are computed in fp64 (a thread each per row and head) and c is kept in two fp32 terms, so that the difference
// of two close ones is as exact as the exponent of a single step, however far the sum has come; C . B runs in 16 chains, S C
// and the update in four.
//
// C . B is the same for all heads of a group: ssm_chunk32_pre computes its lower triangle once, into a workspace,
// and with it the step sizes, whose chain of softplus and sums would hold up every chunk of the scan.
//
// Workgroup of the scan: 8 waves, 32 value columns of one (segment, head).  Waves 0-3 produce the output rows
// [16 w, 16 w + 16) of a chunk: C is in registers, C . B comes from the workspace in the layout that the next product takes.
// Waves 4-7 update the state, whose image for S C is republished in LDS between chunks.  Row wave w has w + 1 tiles of M, so
// state wave 4 + w, which shares its SIMD, has the fewer state tiles the larger w is.  LDS rows are padded so that b128 reads
// along a row and b32 reads of every fourth row both spread over the banks.
//
// In the block of 16 rows on the diagonal a zero weight meets rows that are still to come.  Where one of them is not finite, the
// product would reach back, so that a chunk with such an x runs this block term by term.
//
// Bound by the chain of a chunk (4.3 us of which the products of a SIMD, 152 of 32 cycles each, are 2), as a head has two
// workgroups and 128 heads just fill the chip.  900 rows, 128 heads of 64, state 128: token by token, bound by the issue of
// multiply-adds, 228 us; here 76.  C . B in every workgroup instead: 95; step sizes made by a state wave as well: 86;
// loads behind branches: 89.  Error against fp64 (y / state): a = -exp(1.5 normal) 1.9e-7 / 2.1e-7 token by token, 1.2e-7 /
// 7.4e-8 here; a from -1 to -16 9.4e-8 / 6.4e-8 and 9.1e-8 / 5.8e-8; |a| < 0.02 4.9e-7 / 5.9e-7 and 1.5e-7 / 9.1e-8.
#include "common.h"

namespace {
constexpr int Q = 64, PP = 32, LX = PP + 4;

struct Chunk32Args {
    const float* xbc;
    int ldx;
    ProjSrc u;  // dt columns
    int dt_at;
    const float* dt_bias;
    const float* a_neg;
    const float* d_skip;
    float* state;  // [slots][heads][P][N]
    const int *cu, *slots, *pos0;
    float* y;      // [T][heads * P]
    float* cb;     // [chunks][groups][64][64]: C . B, tiles on and below the diagonal
    float* steps;  // [chunks][heads][4][64]: c in two terms, dt, update weight 2^(c_last - c) dt
    int heads, P, N, groups, seg0;
};

// chunks before the first one of a segment, at most: floor(row / 64) grows by at least the whole chunks of a segment
__device__ __forceinline__ size_t first_chunk(const Chunk32Args& a, int seg) { return a.cu[seg] / Q + (seg - a.seg0); }

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// 2^(ah + al - bh - bl): what the difference of the heads rounds off goes with the tails, to first order
__device__ __forceinline__ float exp2_diff(float ah, float al, float bh, float bl) {
    const float d = ah - bh, back = ah - d;
    const float e = __builtin_amdgcn_exp2f(d);
    return fmaf(e, 0.6931471805599453f * ((back - bh) + (al - bl)), e);
}
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
}  // namespace

// grid (chunks of the longest segment, groups + ceil(heads / 4), segments).  A group: wave w has rows [16 w, 16 w + 16) of
// the chunk; behind the groups a wave has the step sizes of a head.
template <int NN>
__global__ __launch_bounds__(256) void ssm_chunk32_pre_kernel(const Chunk32Args a) {
    constexpr int NS = NN / 16;
    const int grp = blockIdx.y, seg = a.seg0 + blockIdx.z, t0 = a.cu[seg] + Q * blockIdx.x, re = a.cu[seg + 1];
    if (t0 >= re) return;
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (grp >= a.groups) {
        const int head = 4 * (grp - a.groups) + w;
        if (head >= a.heads) return;
        const float raw = proj_at<true>(a.u, min(t0 + lane, re - 1), a.dt_at + head);
        const bool in = t0 + lane < re;  // rows past the end leave the state as it is
        const double z = (double)raw + a.dt_bias[head];
        const double dt = in ? (z > 40. ? z : log1p(exp(z))) : 0.;
        const double an = (double)a.a_neg[head] * 1.4426950408889634;
        // 2^-400 is zero; a total decay must not make differences of infinities, and what is no number stays none
        double c = in ? an * dt : 0.;
        if (c < -400.) c = -400.;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double v = __shfl_up(c, o, 64);
            if (lane >= o) c += v;
        }
        const float ch = (float)c;
        float* o = a.steps + ((first_chunk(a, seg) + blockIdx.x) * a.heads + head) * (4 * Q) + lane;
        o[0] = ch;
        o[Q] = (float)(c - ch);
        o[2 * Q] = (float)dt;
        o[3 * Q] = (float)(exp2(__shfl(c, 63, 64) - c) * dt);
        return;
    }
    const float* bcol = a.xbc + a.heads * a.P + grp * a.N + 4 * g;
    const float* crow = bcol + a.groups * a.N + (size_t)min(t0 + 16 * w + r16, re - 1) * a.ldx;
    f32x4 cf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) cf[s] = 16 * s + 4 * g < a.N ? ld4(crow + 16 * s) : f32x4{0.f, 0.f, 0.f, 0.f};
    float* out = a.cb + ((first_chunk(a, seg) + blockIdx.x) * a.groups + grp) * (Q * Q) + (16 * w + r16) * Q + 4 * g;
    for (int jb = 0; jb <= w; ++jb) {
        const float* brow = bcol + (size_t)min(t0 + 16 * jb + r16, re - 1) * a.ldx;
        f32x4 v[NS], acc[16];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = 16 * s + 4 * g < a.N ? ld4(brow + 16 * s) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * (s & 3) + e] = mma(v[s][e], cf[s][e], acc[4 * (s & 3) + e]);
#pragma unroll
        for (int o = 8; o > 0; o >>= 1)
#pragma unroll
            for (int e = 0; e < o; ++e) acc[e] += acc[e + o];
        *reinterpret_cast<f32x4*>(out + 16 * jb) = acc[0];  // rows j = 16 jb + 4 g + e, column i = 16 w + r16
    }
}

// NN: state columns in LDS (N <= NN); WHOLE: N == NN and P is a multiple of 32
template <int NN, bool WHOLE>
__global__ __launch_bounds__(512, 2) void ssm_chunk32_kernel(const Chunk32Args a) {
    constexpr int LN = NN + 4, NS = NN / 16, BIT = NN / 32;
    // state tiles (16 n x 16 p) of a wave, at most
    constexpr int TILES = NN == 128 ? 5 : 3;
    __shared__ __attribute__((aligned(16))) float sB[Q * LN];
    __shared__ __attribute__((aligned(16))) float sX[Q * LX];
    __shared__ __attribute__((aligned(16))) float sS[PP * LN];
    __shared__ __attribute__((aligned(16))) float s_st[4][Q];  // as `steps`
    __shared__ int s_bad;  // first row of the last chunk with an x that is not finite
    const int p0 = blockIdx.x * PP, head = blockIdx.y, seg = a.seg0 + blockIdx.z;
    const int rb = a.cu[seg], re = a.cu[seg + 1];
    if (rb >= re) return;
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), w = wv & 3;
    const int inner = a.heads * a.P, grp = head / (a.heads / a.groups);
    const float* xcol = a.xbc + head * a.P + p0;
    const float* bcol = a.xbc + inner + grp * a.N;
    const float* ccol = bcol + a.groups * a.N;
    f32x4 breg[BIT], xreg;
    const int xr = tid / 8, xp = 4 * (tid % 8);
    // Rows past the end are read as the last one and stored as zeros.
    // (Loads are unconditional, also behind the last chunk: behind a branch that may have issued some, the compiler waits for
    // all of them, which put a memory latency into every chunk.)
    auto load_chunk = [&](int t0) {
        const float* xs = xcol + (size_t)min(t0 + xr, re - 1) * a.ldx + xp;
        const float* bs[BIT];
#pragma unroll
        for (int i = 0; i < BIT; ++i) {
            const int idx = tid + 512 * i, row = idx / (NN / 4), n = 4 * (idx % (NN / 4));
            bs[i] = bcol + (size_t)min(t0 + row, re - 1) * a.ldx + n;
        }
        if constexpr (WHOLE) {
#pragma unroll
            for (int i = 0; i < BIT; ++i) breg[i] = ld4(bs[i]);
            xreg = ld4(xs);
        } else {
            const int n = 4 * (tid % (NN / 4));  // 512 is a multiple of NN / 4
#pragma unroll
            for (int i = 0; i < BIT; ++i) breg[i] = n < a.N ? ld4(bs[i]) : f32x4{0.f, 0.f, 0.f, 0.f};
            xreg = p0 + xp < a.P ? ld4(xs) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    auto store_chunk = [&](int t0) {
#pragma unroll
        for (int i = 0; i < BIT; ++i) {
            const int idx = tid + 512 * i, row = idx / (NN / 4), n = 4 * (idx % (NN / 4));
            *reinterpret_cast<f32x4*>(sB + row * LN + n) = t0 + row < re ? breg[i] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const f32x4 x = t0 + xr < re ? xreg : f32x4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<f32x4*>(sX + xr * LX + xp) = x;
        const float top = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
        const float nan = (x[0] + x[1]) + (x[2] + x[3]);  // (the maximum drops one)
        if (!(top < INFINITY) || nan != nan) s_bad = t0;
    };
    load_chunk(rb);
    if (tid == 0) s_bad = -1;
    __syncthreads();
    if (wv < 4) {  // output rows
        const float dsk = a.d_skip[head];
        f32x4 cf[NS];
        auto load_c = [&](int t0) {
            const float* row = ccol + (size_t)min(t0 + 16 * w + r16, re - 1) * a.ldx + 4 * g;
            if constexpr (WHOLE) {
#pragma unroll
                for (int s = 0; s < NS; ++s) cf[s] = ld4(row + 16 * s);
            } else {
#pragma unroll
                for (int s = 0; s < NS; ++s) cf[s] = 16 * s + 4 * g < a.N ? ld4(row + 16 * s) : f32x4{0.f, 0.f, 0.f, 0.f};
            }
        };
        const float* cb = a.cb + (first_chunk(a, seg) * a.groups + grp) * (Q * Q) + (16 * w + r16) * Q + 4 * g;
        f32x4 cbt[4];  // tile jb: rows j = 16 jb + 4 g + e, column i = 16 w + r16
        auto load_cb = [&](bool next) {
            if (next) cb += (size_t)a.groups * (Q * Q);
#pragma unroll
            for (int jb = 0; jb < 4; ++jb)
                cbt[jb] = ld4(cb + 16 * min(jb, w));
        };
        load_c(rb);
        load_cb(false);
        store_chunk(rb);
        __syncthreads();
        for (int t0 = rb; t0 < re; t0 += Q) {
            const bool more = t0 + Q < re;
            load_chunk(t0 + Q);
            // the carried state: y^T[p][i] = sum_n S^T[p][n] C[i][n]
            f32x4 y[2];
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) {
                f32x4 acc[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const f32x4 v = ld4(sS + (16 * pb + r16) * LN + 16 * s + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] = mma(v[e], cf[s][e], acc[e]);
                }
                y[pb] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            }
            const float ch = s_st[0][16 * w + r16], cl = s_st[1][16 * w + r16];
            const float ei = exp2_diff(ch, cl, 0.f, 0.f);
            const bool bad = s_bad == t0;
            f32x4 mt[4], my[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            load_c(t0 + Q);
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) {
                const f32x4 jh = ld4(s_st[0] + 16 * jb + 4 * g), jl = ld4(s_st[1] + 16 * jb + 4 * g);
                const f32x4 jd = ld4(s_st[2] + 16 * jb + 4 * g);
                const int lim = 16 * (w - jb) + r16 - 4 * g;  // element e is kept when e <= lim
#pragma unroll
                for (int e = 0; e < 4; ++e) mt[jb][e] = e <= lim ? cbt[jb][e] * (exp2_diff(ch, cl, jh[e], jl[e]) * jd[e]) : 0.f;
            }
            load_cb(more);
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) {
                if (jb > w || (jb == w && bad)) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int pb = 0; pb < 2; ++pb)
                        my[pb] = mma(sX[(16 * jb + 4 * g + e) * LX + 16 * pb + r16], mt[jb][e], my[pb]);
            }
            if (bad) {
                const f32x4 m = w == 0 ? mt[0] : w == 1 ? mt[1] : w == 2 ? mt[2] : mt[3];
#pragma unroll 1
                for (int j0 = 0; j0 < 16; j0 += 4)
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float mj = __shfl(m[k], 4 * j0 + r16, 64);
                        if (j0 + k > r16) continue;
#pragma unroll
                        for (int pb = 0; pb < 2; ++pb) {
                            const f32x4 x = ld4(sX + (16 * w + j0 + k) * LX + 16 * pb + 4 * g);
#pragma unroll
                            for (int e = 0; e < 4; ++e) my[pb][e] = fmaf(mj, x[e], my[pb][e]);
                        }
                    }
            }
            const int t = t0 + 16 * w + r16;  // lane: this row, value columns 16 pb + 4 g .. + 4
            if (t < re) {
#pragma unroll
                for (int pb = 0; pb < 2; ++pb) {
                    const int p = 16 * pb + 4 * g;
                    if (p0 + p < a.P) {
                        const f32x4 x = ld4(sX + (16 * w + r16) * LX + p);
                        f32x4 o;
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = fmaf(dsk, x[e], fmaf(ei, y[pb][e], my[pb][e]));
                        *reinterpret_cast<f32x4*>(a.y + (size_t)t * inner + head * a.P + p0 + p) = o;
                    }
                }
            }
            if (more) {
                __syncthreads();  // every wave is done with this chunk's images
                store_chunk(t0 + Q);
                __syncthreads();
            }
        }
        return;
    }
    const int first = NN == 128 ? (w == 0 ? 0 : 4 * w + 1) : (w == 0 ? 0 : 2 * w + 1);  // 5 4 4 3 and 3 2 2 1
    const int count = NN == 128 ? (w == 0 ? 5 : w == 3 ? 3 : 4) : (w == 0 ? 3 : w == 3 ? 1 : 2);
    float* slot = a.state + ((size_t)a.slots[seg] * a.heads + head) * a.P * a.N;
    const bool cont = a.pos0[seg] > 0;
    // tile k: rows n = 16 (k >> 1) + 4 g + e, column p = 16 (k & 1) + r16
    f32x4 st[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        const int k = first + i, p = 16 * (k & 1) + r16, n = 16 * (k >> 1) + 4 * g;
        st[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (i < count && cont && p0 + p < a.P && n < a.N) st[i] = ld4(slot + (size_t)(p0 + p) * a.N + n);
    }
    auto store_state = [&]() {
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            const int k = first + i;
            if (i < count) *reinterpret_cast<f32x4*>(sS + (16 * (k & 1) + r16) * LN + 16 * (k >> 1) + 4 * g) = st[i];
        }
    };
    // the last wave moves the steps
    const float* steps = a.steps + (first_chunk(a, seg) * a.heads + head) * (4 * Q) + 4 * lane;
    f32x4 sreg = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load_steps = [&](bool next) {
        if (next) steps += (size_t)a.heads * (4 * Q);
        sreg = ld4(steps);
    };
    auto store_steps = [&]() {
        if (w == 3) *reinterpret_cast<f32x4*>(&s_st[0][4 * lane]) = sreg;
    };
    load_steps(false);
    store_chunk(rb);
    store_steps();
    store_state();
    __syncthreads();
    for (int t0 = rb; t0 < re; t0 += Q) {
        const bool more = t0 + Q < re;
        load_chunk(t0 + Q);
        load_steps(more);
        const float dec = exp2_diff(s_st[0][Q - 1], s_st[1][Q - 1], 0.f, 0.f);
        // S^T[n][p] = dec S^T + sum_j B[j][n] (w_j x[j][p])
        f32x4 wx[2][4];
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
            const f32x4 wj = ld4(s_st[3] + 16 * jb + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int pt = 0; pt < 2; ++pt) wx[pt][jb][e] = sX[(16 * jb + 4 * g + e) * LX + 16 * pt + r16] * wj[e];
        }
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            if (i < count) {
                const int k = first + i;
                const float* br = sB + 4 * g * LN + 16 * (k >> 1) + r16;
                f32x4 acc[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int jb = 0; jb < 4; ++jb)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x = k & 1 ? wx[1][jb][e] : wx[0][jb][e];
                        acc[e] = mma(br[(16 * jb + e) * LN], x, acc[e]);
                    }
#pragma unroll
                for (int e = 0; e < 4; ++e) st[i][e] = fmaf(dec, st[i][e], (acc[0][e] + acc[1][e]) + (acc[2][e] + acc[3][e]));
            }
        }
        if (more) {
            __syncthreads();  // every wave is done with this chunk's images
            store_chunk(t0 + Q);
            store_steps();
            store_state();
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        const int k = first + i, p = 16 * (k & 1) + r16, n = 16 * (k >> 1) + 4 * g;
        if (i < count && p0 + p < a.P && n < a.N) *reinterpret_cast<f32x4*>(slot + (size_t)(p0 + p) * a.N + n) = st[i];
    }
}

// Segments [seg0, seg0 + nseg), the longest of max_rows rows.  xbc [T][ldx] fp32, u: fp32 slabs, dt columns at dt_at; ws: fp32
// [T / 64 + nseg + 1] chunks, of groups * 64 * 64 + heads * 4 * 64 values.  P % 4 == 0, N % 4 == 0, N <= 128, ldx % 4 == 0,
// xbc on 16 bytes.
MRSUM_API int mrsum_ssm_chunk32(const void* xbc, int ldx, const void* u, int S, int ld, int T, int dt_at, const float* dt_bias,
                                const float* a_neg, const float* d_skip, float* state, const int* cu, const int* slots,
                                const int* pos0, int seg0, int nseg, int max_rows, float* ws, float* y, int heads, int P, int N,
                                int groups, hipStream_t s) {
    if (T <= 0 || nseg <= 0 || max_rows <= 0) return 0;
    if (!cu || !ws || S < 1 || P <= 0 || N <= 0 || P % 4 || N % 4 || N > 128 || ldx % 4 || (uintptr_t)xbc % 16 || heads <= 0 ||
        groups <= 0 || heads % groups || groups + heads / 4 > 65534 || heads > 65535 || nseg > 65535 || dt_at + heads > ld ||
        ldx < heads * P + 2 * groups * N)
        return (int)hipErrorInvalidValue;
    const Chunk32Args a{(const float*)xbc, ldx, ProjSrc{u, S, (size_t)T * ld, ld}, dt_at, dt_bias, a_neg, d_skip, state,
                        cu, slots, pos0, y, ws, ws + (size_t)(T / Q + nseg + 1) * groups * (Q * Q), heads, P, N, groups, seg0};
    const bool whole = (N == 64 || N == 128) && P % PP == 0;
    const dim3 pre(ceil_div(max_rows, Q), groups + ceil_div(heads, 4), nseg), grid(ceil_div(P, PP), heads, nseg);
    if (N <= 64) {
        ssm_chunk32_pre_kernel<64><<<pre, 256, 0, s>>>(a);
        if (whole) ssm_chunk32_kernel<64, true><<<grid, 512, 0, s>>>(a);
        else ssm_chunk32_kernel<64, false><<<grid, 512, 0, s>>>(a);
    } else {
        ssm_chunk32_pre_kernel<128><<<pre, 256, 0, s>>>(a);
        if (whole) ssm_chunk32_kernel<128, true><<<grid, 512, 0, s>>>(a);
        else ssm_chunk32_kernel<128, false><<<grid, 512, 0, s>>>(a);
    }
    return (int)hipGetLastError();
}
