// Gated delta rule, token by token (decoded tokens; 32-bit models; head sizes the chunked form does not take), with the
// gated head-wise output norm in the same launch; prompt portions have a kernel of their own that stages the rows ahead.  Per head, S [dim][vdim]:
//
//     S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
//     out = o / rms(o) * w * silu(gate)
//
// k, q: the convolved rows divided by sqrt(sum of squares + 1e-6), q also times dim^-1/2; beta = logistic(b),
// g = exp(a_neg softplus(a + dt_bias)), all in fp32.  The state S^T [slots][heads][P][N4] (P = vdim, N = dim, N4: N
// rounded up to 4, zeros past it) is carried in registers; o of the new state comes from the old one as
// g S^T q + (k . q) u, so both products over the state run in one pass.
#include "common.h"
#include "delta.h"

__device__ __forceinline__ float4 in4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 in4(const bf16* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
}

// One block per (head, segment): LPR lanes hold a state row (one value column) as NV float4 each, R rows per lane group.
template <bool PARTS, typename T, int NT, int LPR, int NV, int R>
__global__ __launch_bounds__(NT, R <= 8 ? 4 : 1) void delta_step_kernel(const T* __restrict__ x, DeltaArgs a, SegArgs sg, int seg0,
                                                        float* __restrict__ state, T* __restrict__ out) {
    constexpr int RP = NT / LPR;
    __shared__ float s_o[RP * R];
    __shared__ float red[16];
    const int head = blockIdx.x, seg = seg0 + blockIdx.y, tid = threadIdx.x;
    const int r = tid / LPR, l = tid % LPR;
    const int b = sg.cu ? sg.cu[seg] : seg, e = sg.cu ? sg.cu[seg + 1] : seg + 1;
    float* st = state + ((size_t)sg.slots[seg] * a.heads + head) * a.P * a.N4;
    const bool cont = sg.pos0[seg] > 0;
    const int kh = head / (a.heads / a.kv_heads);
    float4 S[R][NV];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int p = r + RP * i, n = 4 * (l + LPR * v);
            S[i][v] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (cont && p < a.P && n < a.N4) S[i][v] = load_state4(st + (size_t)p * a.N4 + n);
        }
    const bool whole = a.N % 4 == 0 && a.ldx % 4 == 0 && a.xk % 4 == 0;
    const float an = a.a_neg[head], db = a.dt_bias[head];
    for (int t = b; t < e; ++t) {
        const T* row = x + (size_t)t * a.ldx;
        // this thread's output column: gate and weight are read before they are needed
        const int p0 = min(tid, a.P - 1);
        const float z0 = proj_at<PARTS>(a.u, t, a.g_at + head * a.P + p0), w0 = a.norm[p0];
        float q[NV][4], k[NV][4];
        float qq = 0.f, kk = 0.f, kq = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v)
        {
            const int n0 = 4 * (l + LPR * v);
            if (whole) {  // four neighbouring columns at once
                const float4 qv = in4(row + kh * a.N + min(n0, a.N - 4)), kv = in4(row + a.xk + kh * a.N + min(n0, a.N - 4));
                const float on = n0 < a.N ? 1.f : 0.f;
                q[v][0] = on * qv.x; q[v][1] = on * qv.y; q[v][2] = on * qv.z; q[v][3] = on * qv.w;
                k[v][0] = on * kv.x; k[v][1] = on * kv.y; k[v][2] = on * kv.z; k[v][3] = on * kv.w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    q[v][j] = n0 + j < a.N ? (float)row[kh * a.N + n0 + j] : 0.f;
                    k[v][j] = n0 + j < a.N ? (float)row[a.xk + kh * a.N + n0 + j] : 0.f;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                qq += q[v][j] * q[v][j];
                kk += k[v][j] * k[v][j];
                kq += k[v][j] * q[v][j];
            }
        }
        const float beta = logistic(proj_at<PARTS>(a.u, t, a.b_at + head));
        const float g = expf(an * softplus(proj_at<PARTS>(a.u, t, a.a_at + head) + db));
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) {
            qq += __shfl_xor(qq, o, 64);
            kk += __shfl_xor(kk, o, 64);
            kq += __shfl_xor(kq, o, 64);
        }
        const float rk = 1.f / sqrtf(kk + 1e-6f), rq = a.q_scale / sqrtf(qq + 1e-6f);
        constexpr int GR = R < 4 ? R : 4;  // rows reduced together
#pragma unroll
        for (int i0 = 0; i0 < R; i0 += GR) {
            float sk[GR], sq[GR], vv[GR];
#pragma unroll
            for (int i = 0; i < GR; ++i) {
                const int p = r + RP * (i0 + i);
                vv[i] = p < a.P ? (float)row[a.xv + head * a.P + p] : 0.f;
                sk[i] = sq[i] = 0.f;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const float4 w = S[i0 + i][v];
                    sk[i] += w.x * k[v][0] + w.y * k[v][1] + w.z * k[v][2] + w.w * k[v][3];
                    sq[i] += w.x * q[v][0] + w.y * q[v][1] + w.z * q[v][2] + w.w * q[v][3];
                }
            }
#pragma unroll
            for (int o = LPR / 2; o > 0; o >>= 1)
#pragma unroll
                for (int i = 0; i < GR; ++i) {
                    sk[i] += __shfl_xor(sk[i], o, 64);
                    sq[i] += __shfl_xor(sq[i], o, 64);
                }
#pragma unroll
            for (int i = 0; i < GR; ++i) {
                const float u = beta * (vv[i] - g * rk * sk[i]);
                const float uk = u * rk;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    float4& w = S[i0 + i][v];
                    w.x = g * w.x + uk * k[v][0];
                    w.y = g * w.y + uk * k[v][1];
                    w.z = g * w.z + uk * k[v][2];
                    w.w = g * w.w + uk * k[v][3];
                }
                if (l == 0) s_o[r + RP * (i0 + i)] = rq * (g * sq[i] + uk * kq);
            }
        }
        __syncthreads();
        float ss = 0.f;
        for (int p = tid; p < a.P; p += NT) ss += s_o[p] * s_o[p];
        const float inv = 1.f / sqrtf(block_sum(ss, red) / (float)a.P + a.eps);
        T* o = out + (size_t)t * a.ldo + a.col + head * a.P;
        for (int p = tid; p < a.P; p += NT) {
            const float z = p < NT ? z0 : proj_at<PARTS>(a.u, t, a.g_at + head * a.P + p);
            o[p] = (T)(s_o[p] * inv * (p < NT ? w0 : a.norm[p]) * z * logistic_for<T>(z));
        }
        if (head == 0)
            for (int c = a.heads * a.P + tid; c < a.width; c += NT) out[(size_t)t * a.ldo + a.col + c] = (T)0.f;
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int p = r + RP * i, n = 4 * (l + LPR * v);
            if (p < a.P && n < a.N4) store_state4(st + (size_t)p * a.N4 + n, S[i][v]);
        }
}

template <bool PARTS, typename T>
static int launch_delta_step(const void* x, const DeltaArgs& a, const SegArgs& sg, int seg0, int nseg, float* state,
                             void* out, hipStream_t s) {
    const dim3 g(a.heads, nseg);
    const int q = a.N4 / 4;
#define DS(NT, L, V, R_) \
    delta_step_kernel<PARTS, T, NT, L, V, R_><<<g, NT, 0, s>>>((const T*)x, a, sg, seg0, state, (T*)out)
#define DS_R(NT, L, V)                                       \
    {                                                        \
        const int rp = NT / L;                               \
        if (a.P <= rp) DS(NT, L, V, 1);                      \
        else if (a.P <= 2 * rp) DS(NT, L, V, 2);             \
        else if (a.P <= 4 * rp) DS(NT, L, V, 4);             \
        else if (a.P <= 8 * rp) DS(NT, L, V, 8);             \
        else if (a.P <= 16 * rp) DS(NT, L, V, 16);           \
        else return (int)hipErrorInvalidValue;               \
    }
    if (q <= 8) DS_R(256, 8, 1)
    else if (q <= 16) DS_R(256, 16, 1)
    else if (q <= 32 && a.P > 64 && a.P <= 128 && a.heads * nseg <= 256) DS(1024, 32, 1, 4);  // one block per CU
    else if (q <= 32) DS_R(512, 32, 1)
    else if (q <= 64) DS_R(512, 64, 1)
    else return (int)hipErrorInvalidValue;
#undef DS_R
#undef DS
    return (int)hipGetLastError();
}

// Segments [seg0, seg0 + nseg).  P <= 512 up to N = 32, 256 up to 128, 128 up to 256.  x [T][ldx] bf16 / fp32 (x32): convolved q | k | v; u: the projection (b, a and gate
// columns); out rows [T][ldo], columns [col, col + width) (zeros past heads * P).
MRSUM_API int mrsum_delta_step(const void* x, int ldx, int x32, int xk, int xv, const void* u, int S, int ld, int T, int b_at,
                               int a_at, int g_at, const float* dt_bias, const float* a_neg, const float* norm, float eps,
                               float* state, const int* cu, const int* slots, const int* pos0, int seg0, int nseg, void* out,
                               int ldo, int col, int width, int heads, int kv_heads, int P, int N, hipStream_t s) {
    if (T <= 0 || nseg <= 0) return 0;
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || nseg > 65535 || b_at + heads > ld || a_at + heads > ld ||
        g_at + heads * P > ld || ldx < xv + heads * P || xk < kv_heads * N || xv < xk + kv_heads * N ||
        width < heads * P || col + width > ldo || (x32 && S < 1))
        return (int)hipErrorInvalidValue;
    const DeltaArgs a{ProjSrc{u, S, (size_t)T * ld, ld}, b_at, a_at, g_at, dt_bias, a_neg, norm, eps,
                      1.f / sqrtf((float)N), ldx, xk, xv, ldo, col, width, heads, kv_heads, P, N, (N + 3) / 4 * 4};
    const SegArgs sg{cu, nullptr, slots, pos0};
    if (x32) return launch_delta_step<true, float>(x, a, sg, seg0, nseg, state, out, s);
    if (S) return launch_delta_step<true, bf16>(x, a, sg, seg0, nseg, state, out, s);
    return launch_delta_step<false, bf16>(x, a, sg, seg0, nseg, state, out, s);
}

// The same recurrence over longer segments, without the output norm (y: fp32 rows [T - y0][heads * P], row t at t - y0).  A
// (segment, head) is one serial chain of rows: reading each row's operands from memory inside the chain costs a memory
// latency and two block barriers a row.  Here blocks of 16 rows arrive in LDS ahead of their use, keys and queries
// already divided by their lengths; what is left on the chain is one product over the state, a DPP sum and the update.
// 16 lanes hold a state row, R rows (value columns) per lane group; a block has 16 R value columns of one head.
constexpr int PORTION = 16;

template <bool PARTS, typename T, int NV, int R>
__global__ __launch_bounds__(256) void delta_portion_kernel(const T* __restrict__ x, DeltaArgs a, SegArgs sg, int seg0,
                                                            float* __restrict__ state, float* __restrict__ y, int y0) {
    constexpr int NF = 64 * NV, RB = 16 * R;
    __shared__ __attribute__((aligned(16))) float s_kq[2][PORTION][2][NF];
    __shared__ float s_v[2][PORTION][RB];
    __shared__ __attribute__((aligned(16))) float4 s_c[2][PORTION];  // step size, decay, k . q
    const int head = blockIdx.y, seg = seg0 + blockIdx.z, tid = threadIdx.x;
    const int r = tid >> 4, l = tid & 15, p0 = blockIdx.x * RB;
    const int b = sg.cu[seg], e = sg.cu[seg + 1];
    float* st = state + ((size_t)sg.slots[seg] * a.heads + head) * a.P * a.N4;
    const bool cont = sg.pos0[seg] > 0;
    const int kh = head / (a.heads / a.kv_heads);
    const float an = a.a_neg[head], db = a.dt_bias[head];
    const bool whole = a.N % 4 == 0 && a.ldx % 4 == 0 && a.xk % 4 == 0 && (uintptr_t)x % (4 * sizeof(T)) == 0;
    float4 S[R][NV];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int p = p0 + r * R + i, n = 4 * (l + 16 * v);
            S[i][v] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (cont && p < a.P && n < a.N4) S[i][v] = *reinterpret_cast<const float4*>(st + (size_t)p * a.N4 + n);
        }
    // lane group r fetches row r of the block: k, q and R value columns a lane; its first lanes step size and decay
    float4 fk[NV], fq[NV];
    float fv[R], fc = 0.f;
    auto fetch = [&](int t0) {
        const int t = t0 + r;
        const bool in = t < e;
        const T* row = x + (size_t)(in ? t : b) * a.ldx;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int n = 4 * (l + 16 * v);
            fk[v] = row4(row + a.xk + kh * a.N + n, whole, in ? a.N - n : 0);
            fq[v] = row4(row + kh * a.N + n, whole, in ? a.N - n : 0);
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int p = p0 + l + 16 * i;
            fv[i] = in && p < a.P ? (float)row[a.xv + head * a.P + p] : 0.f;
        }
        if (l < 2 && in) fc = proj_at<PARTS>(a.u, t, (l ? a.a_at : a.b_at) + head);
    };
    auto put = [&](int buf, int t0) {
        float kk = 0.f, qq = 0.f, kq = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            kk += fk[v].x * fk[v].x + fk[v].y * fk[v].y + fk[v].z * fk[v].z + fk[v].w * fk[v].w;
            qq += fq[v].x * fq[v].x + fq[v].y * fq[v].y + fq[v].z * fq[v].z + fq[v].w * fq[v].w;
            kq += fk[v].x * fq[v].x + fk[v].y * fq[v].y + fk[v].z * fq[v].z + fk[v].w * fq[v].w;
        }
        kk = sum16(kk); qq = sum16(qq); kq = sum16(kq);
        const float rk = 1.f / sqrtf(kk + 1e-6f), rq = a.q_scale / sqrtf(qq + 1e-6f);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int n = 4 * (l + 16 * v);
            *reinterpret_cast<float4*>(&s_kq[buf][r][0][n]) = make_float4(fk[v].x * rk, fk[v].y * rk, fk[v].z * rk, fk[v].w * rk);
            *reinterpret_cast<float4*>(&s_kq[buf][r][1][n]) = make_float4(fq[v].x * rq, fq[v].y * rq, fq[v].z * rq, fq[v].w * rq);
        }
#pragma unroll
        for (int i = 0; i < R; ++i) s_v[buf][r][l + 16 * i] = fv[i];
        const bool in = t0 + r < e;  // rows past the end leave the state as it is
        const float g = expf(an * softplus(fc + db)), ga = dpp<DPP_XOR1>(g);
        if (l == 0) s_c[buf][r] = make_float4(in ? logistic(fc) : 0.f, in ? ga : 1.f, kq * rk * rq, 0.f);
    };
    fetch(b);
    put(0, b);
    __syncthreads();
    int buf = 0;
    const int yi = l * R / 16, yp = p0 + r * R + yi;  // the value column whose sum this lane ends with
    const bool writes = l % (16 / R) == 0 && yp < a.P;
    for (int t0 = b; t0 < e; t0 += PORTION, buf ^= 1) {
        const bool more = t0 + PORTION < e;
        if (more) fetch(t0 + PORTION);
#pragma unroll 4
        for (int j = 0; j < PORTION; ++j) {
            const float4 c = s_c[buf][j];
            float4 k[NV], q[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                k[v] = *reinterpret_cast<const float4*>(&s_kq[buf][j][0][4 * (l + 16 * v)]);
                q[v] = *reinterpret_cast<const float4*>(&s_kq[buf][j][1][4 * (l + 16 * v)]);
            }
            float sq[R], u[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                float sk = 0.f;
                sq[i] = 0.f;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const float4 w = S[i][v];
                    sk += w.x * k[v].x + w.y * k[v].y + w.z * k[v].z + w.w * k[v].w;
                    sq[i] += w.x * q[v].x + w.y * q[v].y + w.z * q[v].z + w.w * q[v].w;
                }
                u[i] = c.x * (s_v[buf][j][r * R + i] - c.y * sum16(sk));
            }
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    float4& w = S[i][v];
                    w.x = c.y * w.x + u[i] * k[v].x;
                    w.y = c.y * w.y + u[i] * k[v].y;
                    w.z = c.y * w.z + u[i] * k[v].z;
                    w.w = c.y * w.w + u[i] * k[v].w;
                }
            float ui = u[0];
#pragma unroll
            for (int i = 1; i < R; ++i) ui = yi == i ? u[i] : ui;
            const float o = c.y * sum16_scatter<R>(sq, l) + c.z * ui;
            if (writes && t0 + j < e) y[(size_t)(t0 + j - y0) * (a.heads * a.P) + head * a.P + yp] = o;
        }
        if (more) put(buf ^ 1, t0 + PORTION);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int p = p0 + r * R + i, n = 4 * (l + 16 * v);
            if (p < a.P && n < a.N4) *reinterpret_cast<float4*>(st + (size_t)p * a.N4 + n) = S[i][v];
        }
}

template <bool PARTS, typename T>
static int launch_delta_portion(const void* x, const DeltaArgs& a, const SegArgs& sg, int seg0, int nseg, float* state,
                                float* y, int y0, hipStream_t s) {
#define DP(V, R)                                                                                                       \
    delta_portion_kernel<PARTS, T, V, R><<<dim3(ceil_div(a.P, 16 * R), a.heads, nseg), 256, 0, s>>>((const T*)x, a, sg, seg0, \
                                                                                                    state, y, y0)
#define DP_R(V)                                                                     \
    {                                                                               \
        if (r == 1) DP(V, 1);                                                       \
        else if (r == 2) DP(V, 2);                                                  \
        else DP(V, 4);                                                              \
    }
    // as ssm.hip launch_portion: 32 heads of 128 x 128, us at 1 / 2 / 4 rows: one segment of 900 rows (256 blocks)
    // 280 / 339 / 478, four of 1200 (1024) 716 / 626 / 671
    const long long one = (long long)ceil_div(a.P, 16) * a.heads * nseg;  // blocks at one row per lane group
    const int r = one <= 512 ? 1 : one <= 1024 ? 2 : 4;
    if (a.N4 <= 64) DP_R(1)
    else if (a.N4 <= 128) DP_R(2)
    else if (a.N4 <= 256) DP_R(4)
    else return (int)hipErrorInvalidValue;
#undef DP_R
#undef DP
    return (int)hipGetLastError();
}

// Segments [seg0, seg0 + nseg) of several rows each; y [T - y0][heads * P] fp32.  The rest as mrsum_delta_step, which the
// head sizes that it takes come from: a request's prompt is not taken where its decoded tokens would be refused.
MRSUM_API int mrsum_delta_portion(const void* x, int ldx, int x32, int xk, int xv, const void* u, int S, int ld, int T,
                                  int b_at, int a_at, const float* dt_bias, const float* a_neg, float* state,
                                  const int* cu, const int* slots, const int* pos0, int seg0, int nseg, float* y, int y0,
                                  int heads, int kv_heads, int P, int N, hipStream_t s) {
    if (T <= 0 || nseg <= 0) return 0;
    if (!cu || heads <= 0 || heads > 65535 || kv_heads <= 0 || heads % kv_heads || nseg > 65535 || b_at + heads > ld ||
        a_at + heads > ld || ldx < xv + heads * P || xk < kv_heads * N || xv < xk + kv_heads * N || (x32 && S < 1) ||
        P > (N <= 32 ? 512 : N <= 128 ? 256 : 128))
        return (int)hipErrorInvalidValue;
    const DeltaArgs a{ProjSrc{u, S, (size_t)T * ld, ld}, b_at, a_at, 0, dt_bias, a_neg, nullptr, 0.f,
                      1.f / sqrtf((float)N), ldx, xk, xv, 0, 0, 0, heads, kv_heads, P, N, (N + 3) / 4 * 4};
    const SegArgs sg{cu, nullptr, slots, pos0};
    if (x32) return launch_delta_portion<true, float>(x, a, sg, seg0, nseg, state, y, y0, s);
    if (S) return launch_delta_portion<true, bf16>(x, a, sg, seg0, nseg, state, y, y0, s);
    return launch_delta_portion<false, bf16>(x, a, sg, seg0, nseg, state, y, y0, s);
}
