// Chunked state-space scan on MFMA (prompt portions, 16-bit activations): the recurrence of ssm.hip's ssm_step over
// chunks of 64 tokens in matrix form.  With c_i the running sum of a dt over the chunk (fp32, log2 units), per head
//
//   M[i][j] = (C_i . B_j) 2^(c_i - c_j) dt_j  (j <= i)          y_i = sum_j M[i][j] x_j + 2^(c_i) (S C_i) + D x_i
//   S      <- 2^(c_last) S + sum_j 2^(c_last - c_j) dt_j x_j B_j^T
//
// x, B and C are 16-bit operands (exact); everything fp32 that meets them in a product -- M, the state S, the weighted
// x -- enters as TWO bf16 terms (hi + lo, 16 bits of mantissa), accumulated in fp32; the state itself is carried in
// fp32 accumulator registers.
//
// Workgroup: 8 waves, one (work item, head); a work item is a run of rows of one segment.  B and X of a chunk sit
// row-major in LDS (next chunk prefetched in registers); transposed operands come from ds_read_b64_tr_b16.  Waves 0-3
// produce the output rows, [16 w, 16 w + 16) of the chunk each: C of a wave's rows is in registers, and M^T tiles are
// computed in the accumulator layout that is the next product's operand, so M never touches LDS.  Waves 4-7 update the
// state meanwhile, value columns [16 w, 16 w + 16) (+ 64 for PW = 2) each, in accumulator registers; its hi / lo image
// for S C is republished in LDS between chunks (two barriers a chunk, both reached by every wave).
//
// Few (segment, head) pairs cannot fill 256 CUs, so long segments are cut into runs: STATE_ONLY computes every run's
// final state from zero, ssm_combine chains them into each run's starting state, and the full kernel runs all runs in
// parallel.
//
// PW: 64-wide blocks of value columns (vdim <= 64 PW); NB: 32-wide blocks of the state dimension (state <= 32 NB).
#include "common.h"

namespace {
constexpr int Q = 64;
constexpr float LOG2E = 1.4426950408889634f;
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4 lds_s4;

struct ChunkArgs {
    const bf16* xbc;
    int ldx;
    ProjSrc u;  // dt columns
    int dt_at;
    const float* dt_bias;
    const float* a_neg;
    const float* d_skip;
    float* state;      // [slots][heads][P][N4]
    const int* slots;
    const int* pos0;
    const int4* items;  // (segment, first row, end row, last run of its segment)
    float* ws;          // [items][heads][P][N4] run states, or null: one run per segment, starting from its slot
    float* ws_decay;    // [items][heads]
    float* y;           // [T][heads * P]
    int heads, P, N, N4, groups;
};

__device__ __forceinline__ bf16x8 tr8(const bf16* lo, const bf16* hi) {
    const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)lo);
    const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)hi);
    return __builtin_bit_cast(bf16x8, (s8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}));
}

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void split8(const float* v, bf16x8& hi, bf16x8& lo) {
    u32x4 h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint2 t = split2(v[2 * j], v[2 * j + 1]);
        h[j] = t.x;
        l[j] = t.y;
    }
    hi = __builtin_bit_cast(bf16x8, h);
    lo = __builtin_bit_cast(bf16x8, l);
}
}  // namespace

// SCAN_WAVE: a wave that only makes the step sizes; STATE_ONLY, where every other wave updates the state (launch_state).
template <int PW, int NB, bool STATE_ONLY, bool SCAN_WAVE>
__global__ __launch_bounds__(STATE_ONLY ? (SCAN_WAVE ? 320 : 256) : 512,
                             STATE_ONLY ? (PW == 1 && NB == 4 && !SCAN_WAVE ? 4 : 2) : (PW == 1 && NB <= 4 ? 4 : 2)) void
ssm_chunk_kernel(const ChunkArgs a) {
    constexpr int NTH = STATE_ONLY ? 256 : 512;
    constexpr int PP = 64 * PW, NN = 32 * NB;
    constexpr int LB = NN + 16, LX = PP + 16;  // LDS row strides: +32 bytes spreads rows over the banks
    constexpr int NT = 2 * NB;                 // 16-wide state blocks
    constexpr int BIT = (256 * NB + NTH - 1) / NTH, XIT = 512 * PW / NTH;  // staging rounds of B and X
    __shared__ __attribute__((aligned(16))) bf16 sB[Q * LB];
    __shared__ __attribute__((aligned(16))) bf16 sX[Q * LX];
    __shared__ __attribute__((aligned(16))) bf16 sSh[STATE_ONLY ? 8 : PP * LB];
    __shared__ __attribute__((aligned(16))) bf16 sSl[STATE_ONLY ? 8 : PP * LB];
    __shared__ __attribute__((aligned(16))) float s_cum[Q], s_dt[Q], s_w[Q];
    const int head = blockIdx.x, item = blockIdx.y;
    const int4 it = a.items[item];
    const int seg = it.x, rb = it.y, re = it.z;
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), w = wv & 3;
    const bool updates = STATE_ONLY || wv >= 4;  // wave role: state update | output rows
    const int q4 = r16 >> 2, p4 = 4 * (r16 & 3);
    const int inner = a.heads * a.P, grp = head / (a.heads / a.groups);
    const bf16* xcol = a.xbc + head * a.P;
    const bf16* bcol = a.xbc + inner + grp * a.N;
    const bf16* ccol = bcol + a.groups * a.N;
    u32x4 breg[BIT], xreg[XIT];  // staging registers of one chunk
#define LOAD_CHUNK(T0)                                                                                  \
    {                                                                                                   \
        _Pragma("unroll") for (int i = 0; i < BIT; ++i) {                                               \
            const int idx = tid + NTH * i, row = idx / (4 * NB), n = 8 * (idx % (4 * NB));              \
            breg[i] = u32x4{0, 0, 0, 0};                                                                \
            if (row < Q && (T0) + row < re && n < a.N)                                                  \
                breg[i] = *reinterpret_cast<const u32x4*>(bcol + (size_t)((T0) + row) * a.ldx + n);     \
        }                                                                                               \
        _Pragma("unroll") for (int i = 0; i < XIT; ++i) {                                               \
            const int idx = tid + NTH * i, row = idx / (8 * PW), p = 8 * (idx % (8 * PW));              \
            xreg[i] = u32x4{0, 0, 0, 0};                                                                \
            if ((T0) + row < re && p < a.P)                                                             \
                xreg[i] = *reinterpret_cast<const u32x4*>(xcol + (size_t)((T0) + row) * a.ldx + p);     \
        }                                                                                               \
    }
#define STORE_CHUNK()                                                                                   \
    {                                                                                                   \
        _Pragma("unroll") for (int i = 0; i < BIT; ++i) {                                               \
            const int idx = tid + NTH * i, row = idx / (4 * NB), n = 8 * (idx % (4 * NB));              \
            if (row < Q) *reinterpret_cast<u32x4*>(sB + row * LB + n) = breg[i];                        \
        }                                                                                               \
        _Pragma("unroll") for (int i = 0; i < XIT; ++i) {                                               \
            const int idx = tid + NTH * i, row = idx / (8 * PW), p = 8 * (idx % (8 * PW));              \
            *reinterpret_cast<u32x4*>(sX + row * LX + p) = xreg[i];                                     \
        }                                                                                               \
    }
    // The raw step sizes of a chunk become dt, the running sum and the update weights beside the chunk before, in a wave that
    // updates the state (it has half the products of one that makes output rows) or, where all do, in one of its own if SCAN_WAVE:
    // between the chunk's two barriers only their stores are left, and the update weights' one exchange of lanes and
    // exponential.  All of it there made every wave wait for seven exchanges one after the other.
    const float an = a.a_neg[head] * LOG2E, db = a.dt_bias[head];
    float dtr = 0.f, cum = 0.f;
#define LOAD_DT(T0)                                                                                     \
    {                                                                                                   \
        const int ti_ = min((T0) + lane, re - 1);                                                       \
        dtr = a.u.S ? proj_at<true>(a.u, ti_, a.dt_at + head) : proj_at<false>(a.u, ti_, a.dt_at + head); \
    }
#define SCAN_DT(T0)                                                                                     \
    {                                                                                                   \
        dtr = (T0) + lane < re ? softplus(dtr + db) : 0.f;                                              \
        cum = an * dtr;                                                                                 \
        _Pragma("unroll") for (int o = 1; o < 64; o <<= 1) {                                            \
            const float v = __shfl_up(cum, o, 64);                                                      \
            if (lane >= o) cum += v;                                                                    \
        }                                                                                               \
    }
#define STORE_DT()                                                                                      \
    {                                                                                                   \
        s_cum[lane] = cum;                                                                              \
        s_dt[lane] = dtr;                                                                               \
        s_w[lane] = __builtin_amdgcn_exp2f(__shfl(cum, 63, 64) - cum) * dtr;                            \
    }
    if (SCAN_WAVE && wv == 4) {
        LOAD_DT(rb)
        SCAN_DT(rb)
        STORE_DT()
        __syncthreads();
        for (int t0 = rb + Q; t0 < re; t0 += Q) {
            LOAD_DT(t0)
            SCAN_DT(t0)
            __syncthreads();
            STORE_DT()
            __syncthreads();
        }
        return;
    }
    LOAD_CHUNK(rb)
    if (!updates) {
        if constexpr (!STATE_ONLY) {
            const float dsk = a.d_skip[head];
            bf16x8 cf[NB];
#define LOAD_C(T0)                                                                                      \
    {                                                                                                   \
        const int ti_ = (T0) + 16 * w + r16;                                                            \
        _Pragma("unroll") for (int kb = 0; kb < NB; ++kb) {                                             \
            u32x4 v = u32x4{0, 0, 0, 0};                                                                \
            if (ti_ < re && 32 * kb + 8 * g < a.N)                                                      \
                v = *reinterpret_cast<const u32x4*>(ccol + (size_t)ti_ * a.ldx + 32 * kb + 8 * g);      \
            cf[kb] = __builtin_bit_cast(bf16x8, v);                                                     \
        }                                                                                               \
    }
            LOAD_C(rb)
            STORE_CHUNK()
            __syncthreads();
            for (int t0 = rb; t0 < re; t0 += Q) {
                const bool more = t0 + Q < re;
                if (more) LOAD_CHUNK(t0 + Q)
                f32x4 y[4 * PW];
#pragma unroll
                for (int pb = 0; pb < 4 * PW; ++pb) y[pb] = f32x4{0.f, 0.f, 0.f, 0.f};
                // the carried state: y^T[p][i] = sum_n S^T[p][n] C[i][n], then 2^(c_i)
#pragma unroll
                for (int kb = 0; kb < NB; ++kb)
#pragma unroll
                    for (int pb = 0; pb < 4 * PW; ++pb) {
                        const int o = (16 * pb + r16) * LB + 32 * kb + 8 * g;
                        y[pb] = mma(*reinterpret_cast<const bf16x8*>(sSh + o), cf[kb], y[pb]);
                        y[pb] = mma(*reinterpret_cast<const bf16x8*>(sSl + o), cf[kb], y[pb]);
                    }
                const float ci = s_cum[16 * w + r16];
                const float ei = __builtin_amdgcn_exp2f(ci);
#pragma unroll
                for (int pb = 0; pb < 4 * PW; ++pb) y[pb] *= ei;
                // inside the chunk: M^T tiles of two 16-row blocks j at a time are the next product's operand
                for (int jb = 0; jb <= w; jb += 2) {
                    float m[8];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int j0 = 16 * (jb + h);
                        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                        if (jb + h <= w) {
#pragma unroll
                            for (int kb = 0; kb < NB; ++kb)
                                acc = mma(*reinterpret_cast<const bf16x8*>(sB + (j0 + r16) * LB + 32 * kb + 8 * g), cf[kb],
                                          acc);
                        }
                        const float4 cj = *reinterpret_cast<const float4*>(s_cum + j0 + 4 * g);
                        const float4 dj = *reinterpret_cast<const float4*>(s_dt + j0 + 4 * g);
                        const int lim = 16 * w + r16 - (j0 + 4 * g);  // element e is kept when e <= lim
                        m[4 * h + 0] = 0 <= lim ? acc[0] * __builtin_amdgcn_exp2f(ci - cj.x) * dj.x : 0.f;
                        m[4 * h + 1] = 1 <= lim ? acc[1] * __builtin_amdgcn_exp2f(ci - cj.y) * dj.y : 0.f;
                        m[4 * h + 2] = 2 <= lim ? acc[2] * __builtin_amdgcn_exp2f(ci - cj.z) * dj.z : 0.f;
                        m[4 * h + 3] = 3 <= lim ? acc[3] * __builtin_amdgcn_exp2f(ci - cj.w) * dj.w : 0.f;
                    }
                    bf16x8 mh, ml;
                    split8(m, mh, ml);
                    const bf16* xr = sX + (16 * jb + 4 * g + q4) * LX + p4;
#pragma unroll
                    for (int pb = 0; pb < 4 * PW; ++pb) {
                        const bf16x8 xt = tr8(xr + 16 * pb, xr + 16 * LX + 16 * pb);
                        y[pb] = mma(xt, mh, y[pb]);
                        y[pb] = mma(xt, ml, y[pb]);
                    }
                }
                if (more) LOAD_C(t0 + Q)
                // lane: row i = 16 w + r16, value columns 16 pb + 4 g .. + 4
                const int ti = t0 + 16 * w + r16;
                if (ti < re) {
                    float* yr = a.y + (size_t)ti * inner + head * a.P;
#pragma unroll
                    for (int pb = 0; pb < 4 * PW; ++pb) {
                        const int p = 16 * pb + 4 * g;
                        if (p < a.P) {
                            const uint2 xv = *reinterpret_cast<const uint2*>(sX + (16 * w + r16) * LX + p);
                            y[pb][0] += dsk * __uint_as_float(xv.x << 16);
                            y[pb][1] += dsk * __uint_as_float(xv.x & 0xffff0000u);
                            y[pb][2] += dsk * __uint_as_float(xv.y << 16);
                            y[pb][3] += dsk * __uint_as_float(xv.y & 0xffff0000u);
                            *reinterpret_cast<f32x4*>(yr + p) = y[pb];
                        }
                    }
                }
                if (more) {
                    __syncthreads();  // every wave is done with this chunk's LDS images
                    STORE_CHUNK()
                    __syncthreads();
                }
            }
#undef LOAD_C
        }
        return;
    }
    const size_t per_head = (size_t)a.P * a.N4;
    float* slot = a.state + ((size_t)a.slots[seg] * a.heads + head) * per_head;
    float* ws = a.ws ? a.ws + ((size_t)item * a.heads + head) * per_head : nullptr;
    // state tiles: rows n = 16 nb + 4 g + i, column p = 16 w + 64 pw + r16
    f32x4 st[PW][NT];
    {
        const float* src = STATE_ONLY ? nullptr : (ws ? ws : (a.pos0[seg] > 0 ? slot : nullptr));
#pragma unroll
        for (int pw = 0; pw < PW; ++pw)
#pragma unroll
            for (int nb = 0; nb < NT; ++nb) {
                const int p = 64 * pw + 16 * w + r16, n = 16 * nb + 4 * g;
                st[pw][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (src && p < a.P && n < a.N4)
                    st[pw][nb] = *reinterpret_cast<const f32x4*>(src + (size_t)p * a.N4 + n);
            }
    }
#define STORE_STATE()                                                                                   \
    if constexpr (!STATE_ONLY) {                                                                        \
        _Pragma("unroll") for (int pw = 0; pw < PW; ++pw)                                               \
            _Pragma("unroll") for (int nb = 0; nb < NT; ++nb) {                                         \
                const int o = (64 * pw + 16 * w + r16) * LB + 16 * nb + 4 * g;                          \
                const uint2 s01 = split2(st[pw][nb][0], st[pw][nb][1]);                                 \
                const uint2 s23 = split2(st[pw][nb][2], st[pw][nb][3]);                                 \
                *reinterpret_cast<uint2*>(sSh + o) = make_uint2(s01.x, s23.x);                          \
                *reinterpret_cast<uint2*>(sSl + o) = make_uint2(s01.y, s23.y);                          \
            }                                                                                           \
    }
    if (!SCAN_WAVE && w == 0) LOAD_DT(rb)
    STORE_CHUNK()
    if (!SCAN_WAVE && w == 0) {
        SCAN_DT(rb)
        STORE_DT()
    }
    STORE_STATE()
    __syncthreads();
    float total = 0.f;  // STATE_ONLY: the run's summed log2 decay
    for (int t0 = rb; t0 < re; t0 += Q) {
        const bool more = t0 + Q < re;
        if (more) {
            LOAD_CHUNK(t0 + Q)
            if (!SCAN_WAVE && w == 0) LOAD_DT(t0 + Q)
        }
        const float clast = s_cum[Q - 1];
        total += clast;
        // state update: S^T[n][p] = 2^(c_last) S^T + sum_j B[j][n] (w_j x[j][p])
        const float dec = __builtin_amdgcn_exp2f(clast);
#pragma unroll
        for (int pw = 0; pw < PW; ++pw)
#pragma unroll
            for (int nb = 0; nb < NT; ++nb) st[pw][nb] *= dec;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int jr = 32 * kk + 8 * g;
            const float4 w0 = *reinterpret_cast<const float4*>(s_w + jr), w1 = *reinterpret_cast<const float4*>(s_w + jr + 4);
            const float wj[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            bf16x8 xh[PW], xl[PW];
#pragma unroll
            for (int pw = 0; pw < PW; ++pw) {
                const bf16* xr = sX + (jr + q4) * LX + 64 * pw + 16 * w + p4;
                const bf16x8 xv = tr8(xr, xr + 4 * LX);
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = (float)xv[j] * wj[j];
                split8(v, xh[pw], xl[pw]);
            }
            const bf16* br = sB + (jr + q4) * LB + p4;
#pragma unroll
            for (int nb = 0; nb < NT; ++nb) {
                const bf16x8 bt = tr8(br + 16 * nb, br + 4 * LB + 16 * nb);
#pragma unroll
                for (int pw = 0; pw < PW; ++pw) {
                    st[pw][nb] = mma(bt, xh[pw], st[pw][nb]);
                    st[pw][nb] = mma(bt, xl[pw], st[pw][nb]);
                }
            }
        }
        if (more) {
            if (!SCAN_WAVE && w == 0) SCAN_DT(t0 + Q)
            __syncthreads();  // every wave is done with this chunk's LDS images
            if (!SCAN_WAVE && w == 0) STORE_DT()
            STORE_CHUNK()
            STORE_STATE()
            __syncthreads();
        }
    }
#undef LOAD_CHUNK
#undef STORE_CHUNK
#undef LOAD_DT
#undef SCAN_DT
#undef STORE_DT
#undef STORE_STATE
    float* dst = STATE_ONLY ? ws : (it.w ? slot : nullptr);
    if (dst) {
#pragma unroll
        for (int pw = 0; pw < PW; ++pw)
#pragma unroll
            for (int nb = 0; nb < NT; ++nb) {
                const int p = 64 * pw + 16 * w + r16, n = 16 * nb + 4 * g;
                if (p < a.P && n < a.N4) *reinterpret_cast<f32x4*>(dst + (size_t)p * a.N4 + n) = st[pw][nb];
            }
        if (STATE_ONLY && tid == 0) a.ws_decay[(size_t)item * a.heads + head] = __builtin_amdgcn_exp2f(total);
    }
}

// Chain the runs of every segment: ws (each run's final state from zero) becomes each run's STARTING state.
// runs: (segment, first item, items, 0); grid (ceil(per_head / 1024), heads, segments).
__global__ __launch_bounds__(256) void ssm_combine_kernel(const ChunkArgs a, const int4* __restrict__ runs) {
    const int4 r = runs[blockIdx.z];
    const int head = blockIdx.y, per_head = a.P * a.N4;
    const int i = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= per_head) return;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (a.pos0[r.x] > 0)
        s = *reinterpret_cast<const f32x4*>(a.state + ((size_t)a.slots[r.x] * a.heads + head) * per_head + i);
    for (int k = r.y; k < r.y + r.z; ++k) {
        f32x4* p = reinterpret_cast<f32x4*>(a.ws + ((size_t)k * a.heads + head) * per_head + i);
        const f32x4 own = *p;
        *p = s;
        s = a.ws_decay[(size_t)k * a.heads + head] * s + own;
    }
}

namespace {
// The state pass with a wave that only scans has a shorter chain, all passes, us: 64 heads of 64 x 128, 512 workgroups, 134 -> 124, of 64
// x 32, 896 workgroups, 78 -> 73.  But it needs a place for five waves: of states above 128 (185 registers) a CU holds one such workgroup
// and two of four waves, 32 heads, 512 workgroups, 105 and 101, 992 214 and 198; of 64 x 128 three and four, 896 workgroups 135
// and 129, 1000 102 and 97, but 768, three a CU, 111.6 and 111.1.  (Of 128 x 32 three and four too, where both take the same: 896
// workgroups 143 and 140, 1000 98 and 96, but 512 66 and 74.  ssm_runs makes at most 1023.)
template <int PW, int NB>
void launch_state(dim3 grid, const ChunkArgs& a, hipStream_t s) {
    constexpr bool SOME = PW == 1 && NB == 4;
    if constexpr (NB < 8)
        if (!SOME || (long long)grid.x * grid.y <= 768) return ssm_chunk_kernel<PW, NB, true, true><<<grid, 320, 0, s>>>(a);
    if constexpr (NB == 8 || SOME) ssm_chunk_kernel<PW, NB, true, false><<<grid, 256, 0, s>>>(a);
}
}  // namespace

// Rows of the listed runs.  items int4 [n_items], runs int4 [n_runs] with ws / ws_decay when any segment is cut
// (else runs null and n_items = segments).  P % 8 == 0, N % 8 == 0, ldx % 8 == 0; P <= 128, N <= 256 (P <= 64 above
// 128).
MRSUM_API int mrsum_ssm_chunk(const void* xbc, int ldx, const void* u, int S, int ld, int T, int dt_at,
                              const float* dt_bias, const float* a_neg, const float* d_skip, float* state,
                              const int* slots, const int* pos0, const void* items, int n_items, const void* runs,
                              int n_runs, float* ws, float* ws_decay, float* y, int heads, int P, int N, int groups,
                              hipStream_t s) {
    if (T <= 0 || n_items <= 0) return 0;
    if (P <= 0 || N <= 0 || P % 8 || N % 8 || ldx % 8 || P > 128 || N > 256 || (P > 64 && N > 128) || heads % groups ||
        ldx < heads * P + 2 * groups * N || dt_at + heads > ld || n_items > 65535 || n_runs > 65535 || heads > 65535 ||
        (runs && (!ws || !ws_decay)))
        return (int)hipErrorInvalidValue;
    const ChunkArgs a{(const bf16*)xbc, ldx, ProjSrc{u, S, (size_t)T * ld, ld}, dt_at, dt_bias, a_neg, d_skip, state,
                      slots, pos0, (const int4*)items, runs ? ws : nullptr, ws_decay, y, heads, P, N, N, groups};
    const dim3 grid(heads, n_items);
#define CHUNK(PW_, NB_, SO_)                                                              \
    {                                                                                     \
        if constexpr (SO_) launch_state<PW_, NB_>(grid, a, s);                            \
        else ssm_chunk_kernel<PW_, NB_, false, false><<<grid, 512, 0, s>>>(a);            \
    }
#define CHUNK_N(SO_)                                                                          \
    if (P <= 64) {                                                                            \
        if (N <= 32) CHUNK(1, 1, SO_) else if (N <= 64) CHUNK(1, 2, SO_)                      \
        else if (N <= 128) CHUNK(1, 4, SO_) else CHUNK(1, 8, SO_)                             \
    } else {                                                                                  \
        if (N <= 32) CHUNK(2, 1, SO_) else if (N <= 64) CHUNK(2, 2, SO_) else CHUNK(2, 4, SO_) \
    }
    if (runs) {
        CHUNK_N(true)
        ssm_combine_kernel<<<dim3(ceil_div(P * N, 1024), heads, n_runs), 256, 0, s>>>(a, (const int4*)runs);
    }
    CHUNK_N(false)
#undef CHUNK_N
#undef CHUNK
    return (int)hipGetLastError();
}
