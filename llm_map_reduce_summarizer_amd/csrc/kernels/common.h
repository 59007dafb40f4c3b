// Shared helpers for the gfx950 (CDNA4) kernels of mrsum.
//
// Conventions (all kernels):
//   * bf16 tensors are moved as 16-byte vectors (8 x bf16 per lane); scalar
//     bf16 traffic is never used on a hot path (cdna_hip_programming.md G13).
//   * math is fp32; fp32 -> bf16 is a plain cast, which hipcc lowers to
//     v_cvt_pk_bf16_f32 (RNE, NaN-preserving).
//   * wavefront = 64 lanes; every block size is a multiple of 64.
//   * every extern "C" launcher takes raw device pointers + a hipStream_t,
//     never allocates or synchronises (legal inside hipGraph capture) and
//     returns hipGetLastError() as an int.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <math.h>

#define MRSUM_API extern "C" __attribute__((visibility("default")))

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // 16-B staging register (SROA-friendly, unlike HIP's uint4 struct)

static constexpr int WAVE = 64;

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
    return __uint_as_float(bits16 << 16);
}

// 8 packed bf16 (one uint4) -> 8 floats
__device__ __forceinline__ void unpack8(const uint4 v, float* f) {
    f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
    f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
    f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xffff0000u);
    f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xffff0000u);
}

// As a vector: one v_cvt_pk_bf16_f32.  Two 16-bit values put together take one each, and an or.
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(bf16)a, (bf16)b});
}

// two values as bf16 terms (hi, lo): a conversion of both gives either
__device__ __forceinline__ uint2 split2(float x, float y) {
    const uint32_t h = pack2(x, y);
    return make_uint2(h, pack2(x - __uint_as_float(h << 16), y - __uint_as_float(h & 0xffff0000u)));
}

__device__ __forceinline__ uint4 pack8(const float* f) {
    return make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7]));
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Block-wide sum for blockDim.x <= 1024 (uses 16 floats of LDS).
__device__ __forceinline__ float block_sum(float v, float* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    v = wave_sum(v);
    if (lane == 0) red[wid] = v;
    __syncthreads();
    float t = lane < nw ? red[lane] : 0.f;
    t = wave_sum(t);
    __syncthreads();
    return t;
}

// Loads that bypass this CU's L1 (buffer_load ... sc1, aux 16): they read the XCD's L2 / memory copy, so
// a split-K last arriver can read other workgroups' write-through (sc1) stores of THIS launch without an
// agent-scope acquire (buffer_inv sc1 + wait, ~1.7 us) -- the hand-off form of MI355X_MICROARCH.md
// "Valid forms" row 1 / cdna_hip_programming.md Guideline 16: every payload store sc1 and drained before
// the ticket add, the last adder loads after its add returned, the other waves after a barrier, EVERY
// load of the payload such a load.  ``base`` must be wave-uniform (one buffer resource), ``off`` bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sc1_rsrc(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ float4 ld_sc1_f4(__amdgpu_buffer_rsrc_t r, int off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}
__device__ __forceinline__ float2 ld_sc1_f2(__amdgpu_buffer_rsrc_t r, int off) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 16);
    return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
}

// Gated linear unit of the gate_up GEMM epilogues: g sigmoid(alpha g) (u + shift) with g <= limit, |u| <= limit.
// The defaults are SwiGLU.
struct GluArgs {
    float limit = INFINITY, alpha = 1.f, shift = 0.f;
};
__device__ __forceinline__ float glu(float g, float u, const GluArgs& a) {
    g = fminf(g, a.limit);
    u = fminf(fmaxf(u, -a.limit), a.limit);
    return g / (1.f + __expf(-a.alpha * g)) * (u + a.shift);
}

// Attention output form: head h of row t goes to columns [h * pitch, (h + 1) * pitch) of the row, times
// gate[t * gate_ld + h] when a gate is given.
struct AttnEpi {
    const float* gate;
    int gate_ld;
    int pitch;
};

// A projection's result as its consumer kernels read it: fp32 split-K slabs [S][rows][ld] to be summed (PARTS,
// S >= 1), or 16-bit rows [rows][ld].
struct ProjSrc {
    const void* p;
    int S;
    size_t slab;  // elements between slabs
    int ld;
};

template <bool PARTS>
__device__ __forceinline__ float proj_at(const ProjSrc& s, int row, int col) {
    const size_t i = (size_t)row * s.ld + col;
    if constexpr (!PARTS) return (float)reinterpret_cast<const bf16*>(s.p)[i];
    const float* f = reinterpret_cast<const float*>(s.p) + i;
    float a = 0.f;
#pragma unroll 4
    for (int k = 0; k < s.S; ++k) a += f[k * s.slab];
    return a;
}

// 8 (4) consecutive columns; col and ld are multiples of 8 (4)
template <bool PARTS>
__device__ __forceinline__ void proj8(const ProjSrc& s, int row, int col, float* o) {
    const size_t i = (size_t)row * s.ld + col;
    if constexpr (!PARTS) {
        unpack8(*reinterpret_cast<const uint4*>(reinterpret_cast<const bf16*>(s.p) + i), o);
    } else {
        const float* f = reinterpret_cast<const float*>(s.p) + i;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = 0.f;
#pragma unroll 4
        for (int k = 0; k < s.S; ++k) {
            const float4 a = *reinterpret_cast<const float4*>(f + k * s.slab);
            const float4 b = *reinterpret_cast<const float4*>(f + k * s.slab + 4);
            o[0] += a.x; o[1] += a.y; o[2] += a.z; o[3] += a.w;
            o[4] += b.x; o[5] += b.y; o[6] += b.z; o[7] += b.w;
        }
    }
}

template <bool PARTS>
__device__ __forceinline__ float4 proj4(const ProjSrc& s, int row, int col) {
    const size_t i = (size_t)row * s.ld + col;
    if constexpr (!PARTS) {
        const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const bf16*>(s.p) + i);
        return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                           __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
    } else {
        const float* f = reinterpret_cast<const float*>(s.p) + i;
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (int k = 0; k < s.S; ++k) {
            const float4 a = *reinterpret_cast<const float4*>(f + k * s.slab);
            o.x += a.x; o.y += a.y; o.z += a.z; o.w += a.w;
        }
        return o;
    }
}

// A batch as segments, one per sequence: segment i covers rows [cu[i], cu[i + 1]) (cu null: row i) and continues state
// slot slots[i] at absolute position pos0[i].
struct SegArgs {
    const int* cu;       // [n + 1] or null (one row per segment)
    const int* row_seg;  // [T] segment of every row (cu given)
    const int* slots;
    const int* pos0;
};

// The recurrent state of a decoded token: read once, written once.  Nontemporal both ways, it streams: 128 heads of 64 x 128,
// 32 rows (268 MB) 61 -> 53 us, 92 rows 170 -> 136 (5.7 TB/s; either way alone 155 and 167), 8 rows 23 -> 18, one row that
// stays in a cache from token to token 6.3 -> 6.0.
__device__ __forceinline__ float4 load_state4(const float* p) {
    const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
    return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store_state4(float* p, const float4& v) {
    __builtin_nontemporal_store(f32x4{v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4*>(p));
}

__device__ __forceinline__ void load8(const float* p, float* f) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

__device__ __forceinline__ void ld8(const float* p, float* f) { load8(p, f); }
__device__ __forceinline__ void ld8(const bf16* p, float* f) { unpack8(*reinterpret_cast<const uint4*>(p), f); }

// 8 / 4 values to bf16 or fp32 storage (aligned)
__device__ __forceinline__ void store8(bf16* p, const float* f) { *reinterpret_cast<uint4*>(p) = pack8(f); }
__device__ __forceinline__ void store8(float* p, const float* f) {
    reinterpret_cast<float4*>(p)[0] = make_float4(f[0], f[1], f[2], f[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(f[4], f[5], f[6], f[7]);
}
__device__ __forceinline__ void store4(bf16* p, const float4& f) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack2(f.x, f.y), pack2(f.z, f.w));
}
__device__ __forceinline__ void store4(float* p, const float4& f) { *reinterpret_cast<float4*>(p) = f; }

__device__ __forceinline__ float logistic(float x) { return 1.f / (1.f + expf(-x)); }
// logistic for values that leave as 16-bit (T = bf16): hardware exp and reciprocal; accurate for T = float
template <typename T>
__device__ __forceinline__ float logistic_for(float x) {
    if constexpr (sizeof(T) == 2) return __builtin_amdgcn_rcpf(1.f + __expf(-x));
    else return logistic(x);
}
__device__ __forceinline__ float softplus(float x) { return x > 30.f ? x : log1pf(expf(x)); }

// tanh form of gelu: z times the logistic of 2 sqrt(2 / pi) (z + 0.044715 z^3)
template <typename T>
__device__ __forceinline__ float gelu_tanh(float z) {
    return z * logistic_for<T>(1.5957691216057308f * (z + 0.044715f * z * z * z));
}


// bijective XCD remap: blocks b, b+8, ... (one XCD's) get consecutive positions
__device__ __forceinline__ int xcd_position(int bid, int nwg) {
    const int xcd = bid & 7, local = bid >> 3, q = nwg >> 3, r = nwg & 7;
    return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + local;
}

// Sums over aligned groups of 16 lanes without LDS traffic.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;             // quad_perm [1 0 3 2], [2 3 0 1]
constexpr int DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;  // lane i of 8 <- 7 - i, lane i of 16 <- 15 - i
__device__ __forceinline__ float sum16(float v) {
    v += dpp<DPP_MIRROR>(v);
    v += dpp<DPP_HALF_MIRROR>(v);
    v += dpp<DPP_XOR2>(v);
    return v + dpp<DPP_XOR1>(v);
}
// R sums at once: lane l ends with the sum of v[(l & 15) * R / 16]; each exchange halves what is left to add
template <int R>
__device__ __forceinline__ float sum16_scatter(const float (&v)[R], int l) {
    static_assert(R == 1 || R == 2 || R == 4, "rows");
    if constexpr (R == 1) {
        return sum16(v[0]);
    } else {
        const bool hi = l & 8;
        float s;
        if constexpr (R == 4) {
            const float a = (hi ? v[2] : v[0]) + dpp<DPP_MIRROR>(hi ? v[0] : v[2]);
            const float b = (hi ? v[3] : v[1]) + dpp<DPP_MIRROR>(hi ? v[1] : v[3]);
            const bool h4 = l & 4;
            s = (h4 ? b : a) + dpp<DPP_HALF_MIRROR>(h4 ? a : b);
        } else {
            s = (hi ? v[1] : v[0]) + dpp<DPP_MIRROR>(hi ? v[0] : v[1]);
            s += dpp<DPP_HALF_MIRROR>(s);
        }
        s += dpp<DPP_XOR2>(s);
        return s + dpp<DPP_XOR1>(s);
    }
}

// four columns of a bf16 / fp32 row; ``whole``: 4-element aligned, else one by one up to ``n``
template <typename T>
__device__ __forceinline__ float4 row4(const T* p, bool whole, int n) {
    if (n <= 0) return make_float4(0.f, 0.f, 0.f, 0.f);
    if (whole) {
        if constexpr (sizeof(T) == 4) return *reinterpret_cast<const float4*>(p);
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                           __uint_as_float(v.y & 0xffff0000u));
    }
    return make_float4((float)p[0], n > 1 ? (float)p[1] : 0.f, n > 2 ? (float)p[2] : 0.f, n > 3 ? (float)p[3] : 0.f);
}

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Columns [at, at + n) of a projection's slabs through gelu into rows out + t * ldo (n = 0: nothing): a job that kernels
// with few rows take along in blocks of their own.
struct GeluJob {
    int at, n, ldo;
    void* out;
};

template <bool PARTS, typename T>
__device__ __forceinline__ void gelu_piece(const ProjSrc& src, const GeluJob& j, int t, int c) {
    if (c >= j.n) return;
    float v[8];
    proj8<PARTS>(src, t, j.at + c, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = gelu_tanh<T>(v[k]);
    store8(reinterpret_cast<T*>(j.out) + (size_t)t * j.ldo + c, v);
}

// The short causal convolution of a segment of one row t: 4 channels from c on (C in all), whose history it advances.
template <bool PARTS, typename T, int TAPS>
__device__ __forceinline__ void conv_step4(const ProjSrc& src, int at, const float* __restrict__ kernel,
                                           const float* __restrict__ bias, float* __restrict__ state, const SegArgs& sg,
                                           T* __restrict__ out, int C, int t, int c) {
    const bool cont = sg.pos0[t] > 0;
    float* st = state + (size_t)sg.slots[t] * (TAPS - 1) * C + c;
    float4 win[TAPS], kw[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) kw[j] = *reinterpret_cast<const float4*>(kernel + (size_t)j * C + c);
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
        win[j] = *reinterpret_cast<const float4*>(st + (size_t)j * C);
        if (!cont) win[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float4 x = proj4<PARTS>(src, t, at + c);
    if constexpr (PARTS && sizeof(T) == 2)
        x = make_float4((float)(T)x.x, (float)(T)x.y, (float)(T)x.z, (float)(T)x.w);
    win[TAPS - 1] = x;
    float4 a = *reinterpret_cast<const float4*>(bias + c);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        a.x += kw[j].x * win[j].x; a.y += kw[j].y * win[j].y; a.z += kw[j].z * win[j].z; a.w += kw[j].w * win[j].w;
    }
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) *reinterpret_cast<float4*>(st + (size_t)j * C) = win[j + 1];
    a.x *= logistic_for<T>(a.x); a.y *= logistic_for<T>(a.y); a.z *= logistic_for<T>(a.z); a.w *= logistic_for<T>(a.w);
    store4(out + (size_t)t * C + c, a);
}

// ... of all rows and channels, taken along by a kernel with few rows in blocks of its own (C = 0: nothing).
struct ConvJob {
    int at, C;
    const float* kernel;  // [taps][C]
    const float* bias;
    float* state;
    SegArgs sg;
    void* out;  // [T][C]
};

static inline bool gelu_job_ok(const GeluJob& j, int S, int ld) {
    return j.n == 0 || (S >= 1 && j.n > 0 && j.out && j.at >= 0 && j.at % 8 == 0 && j.n % 8 == 0 && j.ldo % 8 == 0 && j.at + j.n <= ld);
}
