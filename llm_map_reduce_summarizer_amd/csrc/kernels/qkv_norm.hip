// Query / key / value preparation of unrotated attention with whole-projection norms.
//
// Per token (one block, the row in registers): q, k, v columns of the input projection (16-bit rows or fp32 split-K slabs) plus
// their biases; q and k divided by the root mean square of the WHOLE projection (all heads at once) and multiplied by
// their weights; q multiplied by the temperature 1 + coef * ln(floor((p + 1) / every) + 1); k and v written into the
// paged cache [pages, G, P, dk | dv] (dk / dv: head widths padded with zeros), q into rows [H][dk], and the head
// gates out_scale * sigmoid(gate column) into fp32 [H].  Everything up to the stores is fp32.
#include "common.h"

struct QkvPrep {
    int H, G, dim, vdim, dk, dv;  // heads, kv heads, head widths, padded widths
    int q, k, v, g;               // first column of each section (multiples of 8); g < 0: no gate
    const float* bias;            // at the projection's columns
    const float* qn;              // [H * dim] or null
    const float* kn;              // [G * dim] or null
    float eps, out_scale, coef, every;  // every <= 0: no temperature
    const int* positions;
    const int* seq_idx;
    const int* block_tables;
    int bt_stride, page;
};

// Two block-wide sums at once (red: 64 floats).
__device__ __forceinline__ float2 block_sum2(float a, float b, float* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) { red[wid] = a; red[32 + wid] = b; }
    __syncthreads();
    return make_float2(wave_sum(lane < nw ? red[lane] : 0.f), wave_sum(lane < nw ? red[32 + lane] : 0.f));
}

template <typename T>
__device__ __forceinline__ void head_store8(T* base, size_t head_stride, int c, int n, int w, const float* f) {
    if (w % 8 == 0) {
        store8(base + (size_t)(c / w) * head_stride + c % w, f);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (c + j < n) base[(size_t)((c + j) / w) * head_stride + (c + j) % w] = (T)f[j];
    }
}

template <typename T>
__device__ __forceinline__ void head_pad(T* base, size_t head_stride, int heads, int w, int wp) {
    const int pad = wp - w;
    for (int i = threadIdx.x; i < heads * pad; i += blockDim.x)
        base[(size_t)(i / pad) * head_stride + w + i % pad] = (T)0.f;
}

// A thread holds CH 8-column pieces of the token's q | k | v columns in registers (sections start at multiples of 8
// and are padded to them, so a piece belongs to one section; the biases of padding columns are zero, and so are the
// projections).
//
// CONV: blocks behind the rows' are those of a convolution of four taps over other columns of the same projection.  Either
// alone is a launch of 5 - 6 us that fills a part of the chip; together they take 6.
template <bool PARTS, typename T, int CH, bool CONV = false>
__global__ __launch_bounds__(1024) void qkv_prep_kernel(ProjSrc src, QkvPrep a, T* __restrict__ q, T* __restrict__ kc,
                                                        T* __restrict__ vc, float* __restrict__ gate, int rows, ConvJob job) {
    __shared__ float red[64];
    const int t = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    if constexpr (CONV) {
        if (t >= rows) {
            const int per = (job.C / 4 + nt - 1) / nt, i = t - rows, c = 4 * (i % per * nt + tid);
            if (c < job.C)
                conv_step4<PARTS, T, 4>(src, job.at, job.kernel, job.bias, job.state, job.sg, (T*)job.out, job.C, i / per, c);
            return;
        }
    }
    const int nq = a.H * a.dim, nk = a.G * a.dim, nv = a.G * a.vdim;
    const int pq = (nq + 7) / 8, pk = (nk + 7) / 8, pieces = pq + pk + (nv + 7) / 8;
    const int pos = a.positions[t];
    const int page = a.block_tables[(size_t)a.seq_idx[t] * a.bt_stride + pos / a.page];
    float v[CH][8];
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int p = tid + nt * i;
        if (p < pieces) {
            const int col = p < pq ? a.q + 8 * p : (p < pq + pk ? a.k + 8 * (p - pq) : a.v + 8 * (p - pq - pk));
            float b[8];
            proj8<PARTS>(src, t, col, v[i]);
            load8(a.bias + col, b);
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                v[i][j] += b[j];
                ss += v[i][j] * v[i][j];
            }
            if (p < pq) sq += ss;
            else if (p < pq + pk) sk += ss;
        }
    }
    const float2 ss = block_sum2(sq, sk, red);
    float qs = a.qn ? 1.f / sqrtf(ss.x / (float)nq + a.eps) : 1.f;
    const float ks = a.kn ? 1.f / sqrtf(ss.y / (float)nk + a.eps) : 1.f;
    if (a.every > 0.f) qs *= 1.f + a.coef * logf(floorf((float)(pos + 1) / a.every) + 1.f);
    T* qo = q + (size_t)t * a.H * a.dk;
    const size_t row = (size_t)page * a.G * a.page + pos % a.page;
    T* ko = kc + row * a.dk;
    T* vo = vc + row * a.dv;
    const size_t hk = (size_t)a.page * a.dk, hv = (size_t)a.page * a.dv;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int p = tid + nt * i;
        if (p >= pieces) continue;
        if (p < pq + pk) {
            const bool isq = p < pq;
            const int c = 8 * (isq ? p : p - pq), n = isq ? nq : nk;
            const float* nw = isq ? a.qn : a.kn;
            const float mul = isq ? qs : ks;
            if (nw && c + 8 <= n) {
                float w[8];
                load8(nw + c, w);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] *= mul * w[j];
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] *= nw && c + j < n ? mul * nw[c + j] : mul;
            }
            if (isq) head_store8(qo, (size_t)a.dk, c, n, a.dim, v[i]);
            else head_store8(ko, hk, c, n, a.dim, v[i]);
        } else {
            head_store8(vo, hv, 8 * (p - pq - pk), nv, a.vdim, v[i]);
        }
    }
    if (a.dk > a.dim) {
        head_pad(qo, (size_t)a.dk, a.H, a.dim, a.dk);
        head_pad(ko, hk, a.G, a.dim, a.dk);
    }
    if (a.dv > a.vdim) head_pad(vo, hv, a.G, a.vdim, a.dv);
    for (int h = tid; h < a.H; h += nt)
        gate[(size_t)t * a.H + h] = a.g >= 0 ? a.out_scale * logistic(proj_at<PARTS>(src, t, a.g + h)) : a.out_scale;
}

template <bool PARTS, typename T>
static int launch_qkv_prep(const ProjSrc& p, const QkvPrep& a, void* q, void* kc, void* vc, float* gate, int rows,
                           const ConvJob& job, hipStream_t s) {
    const int pieces = (a.H * a.dim + 7) / 8 + (a.G * a.dim + 7) / 8 + (a.G * a.vdim + 7) / 8;
    // few rows: one piece per thread (all loads in flight); many rows: 256-thread blocks
    int nt = rows <= 512 ? std::min(1024, ceil_div(pieces, 64) * 64) : 256;
    if (pieces > 8 * nt) nt = 1024;
    const int ch = ceil_div(pieces, nt);
    if (job.C) {
        if (ch > 1) return (int)hipErrorInvalidValue;
        qkv_prep_kernel<PARTS, T, 1, true><<<rows + rows * ceil_div(job.C / 4, nt), nt, 0, s>>>(p, a, (T*)q, (T*)kc, (T*)vc, gate,
                                                                                                rows, job);
        return (int)hipGetLastError();
    }
#define QP(C) qkv_prep_kernel<PARTS, T, C><<<rows, nt, 0, s>>>(p, a, (T*)q, (T*)kc, (T*)vc, gate, rows, job)
    if (ch <= 1) QP(1);
    else if (ch <= 2) QP(2);
    else if (ch <= 3) QP(3);
    else if (ch <= 5) QP(5);
    else if (ch <= 8) QP(8);
    else return (int)hipErrorInvalidValue;
#undef QP
    return (int)hipGetLastError();
}

// src: S = 0 bf16 rows [T][ld], S >= 1 fp32 slabs [S][T][ld].  f32: q / caches fp32 (slabs only), else bf16.
// conv_n > 0: the convolution (as mrsum_conv_silu, four taps, one row per segment) of as many columns from conv_at on
// besides; at most 512 rows and 8192 columns of q, k and v then.
MRSUM_API int mrsum_qkv_prep(const void* src, int S, int ld, int T, int f32, void* q, void* kc, void* vc, float* gate,
                             int H, int G, int dim, int vdim, int dk, int dv, int cq, int ck, int cv, int cg,
                             const float* bias, const float* qn, const float* kn, float eps, float out_scale,
                             float coef, float every, const int* positions, const int* seq_idx, const int* block_tables,
                             int bt_stride, int page, int conv_at, int conv_n, const float* kernel, const float* conv_bias,
                             float* state, const int* slots, const int* pos0, void* conv_out, hipStream_t s) {
    if (T <= 0) return 0;
    if (conv_n < 0 || (conv_n && (T > 512 || conv_n % 8 || conv_at % 8 || conv_at < 0 || conv_at + conv_n > ld || !kernel ||
                                  !conv_bias || !state || !slots || !pos0 || !conv_out)))
        return (int)hipErrorInvalidValue;
    if (H <= 0 || G <= 0 || H % G || dk < dim || dv < vdim || dk % 8 || dv % 8 || (cq | ck | cv) % 8 || ld % 8 ||
        page <= 0 || (f32 && S < 1))
        return (int)hipErrorInvalidValue;
    const QkvPrep a{H, G, dim, vdim, dk, dv, cq, ck, cv, cg, bias, qn, kn, eps, out_scale, coef, every,
                    positions, seq_idx, block_tables, bt_stride, page};
    const ProjSrc p{src, S, (size_t)T * ld, ld};
    const ConvJob job{conv_at, conv_n, kernel, conv_bias, state, SegArgs{nullptr, nullptr, slots, pos0}, conv_out};
    if (f32) return launch_qkv_prep<true, float>(p, a, q, kc, vc, gate, T, job, s);
    if (S) return launch_qkv_prep<true, bf16>(p, a, q, kc, vc, gate, T, job, s);
    return launch_qkv_prep<false, bf16>(p, a, q, kc, vc, gate, T, job, s);
}
