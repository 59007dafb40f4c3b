// Row attention over the paged cache for any head width and value width, in bf16 or fp32 storage with fp32
// arithmetic throughout: one wave, or a few, per (row, query head).  Every lane scores one key of a 64-key page; the
// softmax is online across pages; the value sum runs with the lanes over the value columns.  It serves fp32 models and
// heads the MFMA kernels do not take (attn_prefill.hip / attn_decode.hip / latent_attn.hip): decoded tokens and short
// prompt portions here, long ones in the tiled kernel below; latent attention runs both with the cached rows as keys and
// their first columns as values.
#include "common.h"

constexpr int ROW_PAGE = 64;
constexpr int ROW_MAXV = 8;  // value columns per lane: value widths up to 512

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4(const bf16* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
}

// W waves share one (row, head): wave i walks pages i, i + W, ...; their sums meet in LDS (W 4: one workgroup per head, W 8
// and 16: likewise with more waves; W 1: four heads a workgroup).  A wave's walk is a chain of loads, so few (row, head)
// pairs leave the chip idle: 3 rows of 32 fp32 heads of 128 over 2000 keys took 389 us on one wave each, 56 on 16.
template <typename T, int W>
__global__ __launch_bounds__(W > 4 ? 64 * W : 256) void attn_rows_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc, const int* __restrict__ positions,
    const int* __restrict__ seq_idx, const int* __restrict__ block_tables, int bt_stride, int H, int G, int dk, int dv,
    int ldv, int pitch, float scale, const float* __restrict__ gate, T* __restrict__ out, int out_stride) {
    constexpr int HPB = W > 4 ? 1 : 4 / W;  // heads of a workgroup
    extern __shared__ float sm[];           // q [HPB][dk], p [waves][64]; W > 1: sums [waves][dv], (maximum, sum) [waves]
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, part = wv % W;
    const int t = blockIdx.x, h = blockIdx.y * HPB + wv / W;
    const bool live = h < H;
    if (W == 1 && !live) return;
    float* sq = sm + wv / W * dk;
    float* sp = sm + HPB * dk + wv * ROW_PAGE;
    const T* qr = q + ((size_t)t * H + (live ? h : 0)) * dk;
    if (W == 1) {
        for (int d = lane; d < dk; d += 64) sq[d] = (float)qr[d];  // q and K are zero past the head's width
        __builtin_amdgcn_wave_barrier();
    } else {
        for (int d = 64 * part + lane; d < dk; d += 64 * W) sq[d] = (float)qr[d];
        __syncthreads();
    }
    const int pos = live ? positions[t] : -1, g = (live ? h : 0) / (H / G);
    const int* bt = block_tables + (size_t)seq_idx[t] * bt_stride;
    float m = -INFINITY, l = 0.f, acc[ROW_MAXV];
#pragma unroll
    for (int j = 0; j < ROW_MAXV; ++j) acc[j] = 0.f;
    for (int k0 = part * ROW_PAGE; k0 <= pos; k0 += W * ROW_PAGE) {
        const size_t slab = ((size_t)bt[k0 / ROW_PAGE] * G + g) * ROW_PAGE;
        float s = -INFINITY;
        if (k0 + lane <= pos) {
            const T* kr = kc + (slab + lane) * dk;
            s = 0.f;
            for (int d = 0; d < dk; d += 4) {
                const float4 a = *reinterpret_cast<const float4*>(sq + d), b = ld4(kr + d);
                s += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
            }
            s *= scale;
        }
        const float mn = fmaxf(m, wave_max(s));
        // while all scores are minus infinity there is no weight yet (-inf - -inf would be NaN)
        const float ref = mn == -INFINITY ? 0.f : mn;
        const float alpha = expf(m - ref), p = expf(s - ref);
        m = mn;
        l = l * alpha + wave_sum(p);
        __builtin_amdgcn_wave_barrier();
        sp[lane] = p;
        __builtin_amdgcn_wave_barrier();
        const int n = min(ROW_PAGE, pos + 1 - k0);
#pragma unroll
        for (int j = 0; j < ROW_MAXV; ++j) {
            const int d = lane + 64 * j;
            if (d < dv) {
                float a = acc[j] * alpha;
                const T* vr = vc + slab * ldv + d;
                for (int i = 0; i < n; ++i) a += sp[i] * (float)vr[(size_t)i * ldv];
                acc[j] = a;
            }
        }
    }
    if constexpr (W > 1) {
        constexpr int WAVES = HPB * W;
        float* so = sm + HPB * dk + WAVES * ROW_PAGE;
        float* sml = so + WAVES * dv;
#pragma unroll
        for (int j = 0; j < ROW_MAXV; ++j)
            if (lane + 64 * j < dv) so[wv * dv + lane + 64 * j] = acc[j];
        if (lane == 0) {
            sml[2 * wv] = m;
            sml[2 * wv + 1] = l;
        }
        __syncthreads();
        if (!live) return;
        const int w0 = wv - part;
        float top = -INFINITY, sum = 0.f, f[W];
#pragma unroll
        for (int i = 0; i < W; ++i) top = fmaxf(top, sml[2 * (w0 + i)]);
#pragma unroll
        for (int i = 0; i < W; ++i) {
            f[i] = expf(sml[2 * (w0 + i)] - top);
            sum += f[i] * sml[2 * (w0 + i) + 1];
        }
        const float scl = (gate ? gate[(size_t)t * H + h] : 1.f) / sum;
        T* o = out + (size_t)t * out_stride + (size_t)h * pitch;
        for (int d = 64 * part + lane; d < pitch; d += 64 * W) {
            float v = 0.f;
#pragma unroll
            for (int i = 0; i < W; ++i) v += f[i] * so[(w0 + i) * dv + d];
            o[d] = (T)(v * scl);
        }
        return;
    }
    const float f = (gate ? gate[(size_t)t * H + h] : 1.f) / l;
    T* o = out + (size_t)t * out_stride + (size_t)h * pitch;
#pragma unroll
    for (int j = 0; j < ROW_MAXV; ++j) {
        const int d = lane + 64 * j;
        if (d < pitch) o[d] = (T)(acc[j] * f);
    }
}

// q [T][H][dk], caches [pages][G][64][dk | ldv] (values: the first dv columns of a row; the value rows may be the key
// rows), out rows: head h at columns [h * pitch, (h + 1) * pitch), pitch <= dv.  gate null: ones.
MRSUM_API int mrsum_attn_rows(const void* q, const void* kc, const void* vc, const int* positions, const int* seq_idx,
                              const int* block_tables, int bt_stride, int T, int H, int G, int dk, int dv, int ldv,
                              int pitch, float scale, const float* gate, void* out, int out_stride, int f32,
                              hipStream_t s) {
    if (T <= 0) return 0;
    if (H % G || dk % 4 || pitch > dv || dv > 64 * ROW_MAXV || ldv < dv) return (int)hipErrorInvalidValue;
    if (4 * (dk + ROW_PAGE) * sizeof(float) > 64 * 1024) return (int)hipErrorInvalidValue;
    // Waves per (row, head), from 4 to 8192 pairs of four head shapes over 60 to 6000 keys.  One wave against 16 at 256 pairs:
    // 388 and 52 us (fp32 heads of 128, 2000 keys), 1028 and 172 (latents); 8 against 16 at 512: 101 and 110; 4 against 8 at
    // 1024: 238 and 243, one wave 555.  From 2048 the chip is full: 163 against one wave's 198 for the former at 600 keys,
    // but 484 against 460 for latents, and more at 60 keys.
    const size_t pairs = (size_t)T * H;
    const int waves = pairs <= 256 ? 16 : pairs <= 512 ? 8 : pairs <= 1024 ? 4 : 1;
#define ROWS(T_, W_)                                                                                                   \
    {                                                                                                                  \
        constexpr int HPB = W_ > 4 ? 1 : 4 / W_, WAVES = HPB * W_;                                                     \
        const size_t lds = (HPB * dk + WAVES * (ROW_PAGE + (W_ > 1 ? dv + 2 : 0))) * sizeof(float);                    \
        attn_rows_kernel<T_, W_><<<dim3(T, ceil_div(H, HPB)), 64 * WAVES, lds, s>>>(                                   \
            (const T_*)q, (const T_*)kc, (const T_*)vc, positions, seq_idx, block_tables, bt_stride, H, G, dk, dv,     \
            ldv, pitch, scale, gate, (T_*)out, out_stride);                                                            \
        return (int)hipGetLastError();                                                                                 \
    }
#define FORMS(T_)                   \
    if (waves == 16) ROWS(T_, 16)   \
    if (waves == 8) ROWS(T_, 8)     \
    if (waves == 4) ROWS(T_, 4)     \
    ROWS(T_, 1)
    if (f32) {
        FORMS(float)
    }
    FORMS(bf16)
#undef FORMS
#undef ROWS
}

// ------------------------------------------------------------------------------------------------ prompt portions
// The same attention for many rows of few sequences, on the fp32 matrix instruction.  The row kernel reads every key
// from memory for every (row, head): 1018 us for 900 rows of 32 heads of 128 over 8 kv heads, 4390 over 576-wide latents.
// Here (107 and 508 us; bound by the chain of the block with the most keys: 5 us a tile of which its products are 1.7 where one
// group of waves walks it, 8 us for two tiles at once where two do, 9 us for one of 16 latents) 64
// (row, head) pairs -- RB consecutive rows of HB heads of one kv head -- share key and value tiles of 32 in LDS (two buffers,
// the next tile on its way in registers), a wave for 16 pairs.  With the page ids read when a tile is fetched, its loads
// behind tests of the row and two barriers a tile, 183 and 758 (16-bit caches 201 and 915, now 111 and 561).
//
// Scores are computed transposed, S^T = K Q^T: lane (pair = lane & 15, g = lane >> 4) holds the scores of keys 4 g .. 4 g
// + 3 of a 16-key block, which is how the second product O^T = V^T P^T takes its right operand, so weights stay in
// registers, in fp32.  Every sequence that has rows in the block is a run of its own over the same accumulators.  Tile
// rows are padded by 4 floats (conflict-free b128 key reads and value reads).
// Forms (NQ, NV: 16-column steps of keys and values; SHARED: values are the keys' first columns): KT 32, but 16 where 36 + 32
// steps leave no registers for a larger tile on its way.
// KS 2: two groups of four waves take the tiles in turn, with buffers and sums of their own that meet in LDS at the end, so that
// the block with the most keys walks half of them.  They take the place of two workgroups of a CU (8 us for a tile each where one
// alone takes 5).  900 rows, 32 / 8 heads of 128 in fp32: 158 us, by the order of the blocks 143 - 148, with two groups 107 - 112; error
// against fp64 6.7e-7 and 5.4e-7.  When: ops/hip.py portion_groups.
template <typename T, int NQ, int NV, bool SHARED, int KT, int KS>
__global__ __launch_bounds__(256 * KS, NQ <= 8 ? 2 : 1) void attn_portion_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc, const int* __restrict__ positions,
    const int* __restrict__ seq_idx, const int* __restrict__ block_tables, int bt_stride, int rows, int H, int G, int dk,
    int dv, int ldv, int pitch, float scale, const float* __restrict__ gate, T* __restrict__ out, int out_stride, int HB,
    int RB) {
    constexpr int LK = NQ * 16 + 4, LV = SHARED ? LK : NV * 16 + 4;
    constexpr int TPR = 256 / KT, FK = (NQ * 4 + TPR - 1) / TPR, FV = SHARED ? 1 : (NV * 4 + TPR - 1) / TPR;
    __shared__ __attribute__((aligned(16))) float s_ks[KS][2][KT][LK];
    __shared__ __attribute__((aligned(16))) float s_vs[KS][SHARED ? 1 : 2][SHARED ? 1 : KT][LV];
    __shared__ int s_bads[KS][3];  // tile i (slot i % 3, of SHARED i % 2) holds a value that is not finite
    const int tid = threadIdx.x & 255, part = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int lane = tid & 63, j16 = lane & 15, g4 = lane >> 4;
    auto& s_k = s_ks[part];
    auto& s_v = s_vs[part];
    auto& s_bad = s_bads[part];
    // The last rows, with the most keys, of all heads first.  (All rows of a head first left the later heads' longest walks to begin
    // behind the first one's short ones.)
    const int gh = H / G, hblocks = (gh + HB - 1) / HB, per = G * hblocks, y = blockIdx.x % per, g = y / hblocks, h0 = y % hblocks * HB;
    const int t0 = (gridDim.x / per - 1 - blockIdx.x / per) * RB, tend = min(rows, t0 + RB);
    const int pair = 16 * (tid >> 6) + j16, trow = t0 + pair / HB, hh = h0 + pair % HB;
    const bool valid = pair < RB * HB && trow < tend && hh < gh;
    const int t = valid ? trow : t0, head = g * gh + (valid ? hh : h0), pos = positions[t];
    float4 qf[NQ];
#pragma unroll
    for (int r = 0; r < NQ; ++r) {
        const int c = 16 * r + 4 * g4;
        qf[r] = valid && c < dk ? ld4(q + ((size_t)t * H + head) * dk + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float m = -INFINITY, l = 0.f;
    f32x4 o[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};

    // tile loads: TPR threads a row, four columns each at a time
    const int lr = tid / TPR, lc = 4 * (tid % TPR);
    float4 fk[FK], fv[FV];
    for (int a = t0; a < tend;) {
        const int seq = seq_idx[a];
        int b = a + 1, last = positions[a];
        while (b < tend && seq_idx[b] == seq) last = max(last, positions[b++]);
        if (last < 0) {  // no key for any of these rows: nothing of theirs is read
            a = b;
            continue;
        }
        const bool mine = valid && t >= a && t < b;
        const int* bt = block_tables + (size_t)seq * bt_stride;
        // keys past the last one are read as that (masked), columns past the row as its end and zeroed on the way into LDS
        int page = bt[min(part * KT + lr, last) / ROW_PAGE];  // of this thread's row of the tile fetched next
        auto fetch = [&](int k0) {
            const int key = min(k0 + lr, last);
            const size_t slab = ((size_t)page * G + g) * ROW_PAGE + key % ROW_PAGE;
            page = bt[min(k0 + KS * KT + lr, last) / ROW_PAGE];
#pragma unroll
            for (int i = 0; i < FK; ++i) fk[i] = ld4(kc + slab * dk + min(lc + 4 * TPR * i, dk - 4));
            if constexpr (!SHARED) {
#pragma unroll
                for (int i = 0; i < FV; ++i) fv[i] = ld4(vc + slab * ldv + min(lc + 4 * TPR * i, dv - 4));
            }
        };
        auto put = [&](int buf, int slot) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < FK; ++i) {
                if (lc + 4 * TPR * i >= dk) fk[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (lc + 4 * TPR * i < NQ * 16) *reinterpret_cast<float4*>(&s_k[buf][lr][lc + 4 * TPR * i]) = fk[i];
                if (SHARED && lc + 4 * TPR * i < dv) bad |= !(fabsf(fk[i].x) + fabsf(fk[i].y) + fabsf(fk[i].z) + fabsf(fk[i].w) < INFINITY);
            }
            if constexpr (!SHARED) {
#pragma unroll
                for (int i = 0; i < FV; ++i) {
                    if (lc + 4 * TPR * i >= dv) fv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (lc + 4 * TPR * i < NV * 16) *reinterpret_cast<float4*>(&s_v[buf][lr][lc + 4 * TPR * i]) = fv[i];
                    bad |= !(fabsf(fv[i].x) + fabsf(fv[i].y) + fabsf(fv[i].z) + fabsf(fv[i].w) < INFINITY);
                }
            }
            if (bad) s_bad[slot] = 1;
        };
        if (tid < 3) s_bad[tid] = 0;
        fetch(part * KT);
        __syncthreads();
        put(0, 0);
        __syncthreads();
        // (a group's last tile may be behind the last key: all of it is masked then)
        for (int k0 = part * KT, buf = 0, slot = 0; k0 - part * KT <= last; k0 += KS * KT, buf ^= 1) {
            const bool more = k0 - part * KT + KS * KT <= last;
            if (more) fetch(k0 + KS * KT);
            f32x4 s[KT / 16];
#pragma unroll
            for (int kb = 0; kb < KT / 16; ++kb) s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < NQ; ++r) {
                if (16 * r >= dk) break;
                float4 kf[KT / 16];
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb)
                    kf[kb] = *reinterpret_cast<const float4*>(&s_k[buf][16 * kb + j16][16 * r + 4 * g4]);
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb].x, qf[r].x, s[kb], 0, 0, 0);
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb].y, qf[r].y, s[kb], 0, 0, 0);
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb].z, qf[r].z, s[kb], 0, 0, 0);
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb].w, qf[r].w, s[kb], 0, 0, 0);
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < KT / 16; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[kb][i] = mine && k0 + 16 * kb + 4 * g4 + i <= pos ? s[kb][i] * scale : -INFINITY;
                    mx = fmaxf(mx, s[kb][i]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m, mx), alpha = mn == m ? 1.f : expf(m - mn);
            const float ref = mn == -INFINITY ? 0.f : mn;  // no weight yet, as in the row kernel
            m = mn;
            l *= alpha;
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int c = 0; c < NV; ++c) o[c] *= alpha;
            }
#pragma unroll
            for (int kb = 0; kb < KT / 16; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x = s[kb][i];
                    s[kb][i] = mine && k0 + 16 * kb + 4 * g4 + i <= pos ? expf(x - ref) : 0.f;
                    l += s[kb][i];
                }
            auto vrow = [&](int k) -> const float* { return SHARED ? s_k[buf][k] : s_v[SHARED ? 0 : buf][SHARED ? 0 : k]; };
            if (!s_bad[SHARED ? buf : slot]) {
#pragma unroll
                for (int kb = 0; kb < KT / 16; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float* v = vrow(16 * kb + 4 * g4 + i) + j16;
#pragma unroll
                        for (int c = 0; c < NV; ++c) {
                            if (16 * c >= dv) break;
                            o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[16 * c], s[kb][i], o[c], 0, 0, 0);
                        }
                    }
            } else {  // a later key's infinity times a weight of zero would be no number: only keys that count
                for (int k = 0; k < KT; ++k) {
                    float p = 0.f;
#pragma unroll
                    for (int kb = 0; kb < KT / 16; ++kb)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float x = __shfl(s[kb][i], j16 + 16 * ((k >> 2) & 3), 64);
                            if (k >> 4 == kb && (k & 3) == i) p = x;
                        }
                    if (mine && k0 + k <= pos)
#pragma unroll
                        for (int c = 0; c < NV; ++c)
                            if (16 * c < dv)
#pragma unroll
                                for (int i = 0; i < 4; ++i) o[c][i] += p * vrow(k)[16 * c + 4 * g4 + i];
                }
            }
            if constexpr (SHARED) {  // (registers are full there: the form below spills)
                if (tid == 0) s_bad[buf ^ 1] = 0;
                __syncthreads();
                if (more) put(buf ^ 1, buf ^ 1);
            } else {  // the other buffer and the slot after the next were last read before the barrier ahead of this tile
                const int next = slot == 2 ? 0 : slot + 1;
                if (more) put(buf ^ 1, next);
                if (tid == 0) s_bad[3 - slot - next] = 0;
                slot = next;
            }
            __syncthreads();
        }
        a = b;
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if constexpr (KS == 2) {  // the second group's sums: a piece of 16 bytes a thread at a time, behind the last tile's barrier
        static_assert(NV * 4 * 256 <= 2 * KT * LK && 2 * 256 <= (SHARED ? 1 : 2) * (SHARED ? 1 : KT) * LV, "LDS");
        f32x4* so = reinterpret_cast<f32x4*>(&s_ks[1][0][0][0]);
        float2* sml = reinterpret_cast<float2*>(&s_vs[1][0][0][0]);
        if (part) {
#pragma unroll
            for (int c = 0; c < NV; ++c) so[256 * c + tid] = o[c];
            sml[tid] = make_float2(m, l);
        }
        __syncthreads();
        if (part) return;
        const float2 other = sml[tid];
        const float top = fmaxf(m, other.x), ref = top == -INFINITY ? 0.f : top;
        const float f0 = expf(m - ref), f1 = expf(other.x - ref);
        l = l * f0 + other.y * f1;
#pragma unroll
        for (int c = 0; c < NV; ++c) o[c] = o[c] * f0 + so[256 * c + tid] * f1;
    }
    if (!valid) return;
    const float f = (gate ? gate[(size_t)t * H + head] : 1.f) / l;
    T* dst = out + (size_t)t * out_stride + (size_t)head * pitch;
#pragma unroll
    for (int c = 0; c < NV; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 16 * c + 4 * g4 + i;
            if (d < pitch) dst[d] = (T)(o[c][i] * f);
        }
}

template <typename T>
static int launch_portions(const void* q, const void* kc, const void* vc, const int* positions, const int* seq_idx,
                           const int* block_tables, int bt_stride, int rows, int H, int G, int dk, int dv, int ldv, int pitch,
                           float scale, const float* gate, void* out, int out_stride, int ks, hipStream_t s) {
    const int gh = H / G, HB = std::min(gh, 32), RB = 64 / HB;
    const int grid = ceil_div(rows, RB) * G * ceil_div(gh, HB);
#define AP(NQ, NV, SH, KT, KS)                                                                                           \
    attn_portion_kernel<T, NQ, NV, SH, KT, KS><<<grid, 256 * KS, 0, s>>>((const T*)q, (const T*)kc, (const T*)vc, positions, seq_idx,  \
                                                            block_tables, bt_stride, rows, H, G, dk, dv, ldv, pitch,      \
                                                            scale, gate, (T*)out, out_stride, HB, RB)
    if (dk <= 64 && dv <= 64) {
        if (ks == 2) AP(4, 4, false, 32, 2);
        else AP(4, 4, false, 32, 1);
    } else if (dk <= 128 && dv <= 128) {
        if (ks == 2) AP(8, 8, false, 32, 2);
        else AP(8, 8, false, 32, 1);
    } else if (dk <= 256 && dv <= 256) AP(16, 16, false, 32, 1);
    else if (kc == vc && ldv == dk && dk <= 576 && dv <= 512) AP(36, 32, true, 16, 1);
    else return (int)hipErrorInvalidValue;
#undef AP
    return (int)hipGetLastError();
}

// Arguments as mrsum_attn_rows; widths multiples of 4, rows 16-byte (fp32) or 8-byte (bf16) aligned, and up to 256 wide, or
// up to 576 / 512 where the values are the first columns of the keys.  ks: groups that share a block's keys (2: rows up to 128
// wide; wider ones have one).
MRSUM_API int mrsum_attn_portions(const void* q, const void* kc, const void* vc, const int* positions, const int* seq_idx,
                                  const int* block_tables, int bt_stride, int T, int H, int G, int dk, int dv, int ldv,
                                  int pitch, float scale, const float* gate, void* out, int out_stride, int f32, int ks,
                                  hipStream_t s) {
    if (T <= 0) return 0;
    if (G <= 0 || H % G || dk % 4 || dv % 4 || ldv % 4 || pitch > dv || ldv < dv || G * ceil_div(H / G, 32) > 65535 ||
        (long long)T * H > 0x7fffffff || (ks != 1 && ks != 2))
        return (int)hipErrorInvalidValue;
    if (f32)
        return launch_portions<float>(q, kc, vc, positions, seq_idx, block_tables, bt_stride, T, H, G, dk, dv, ldv, pitch,
                                      scale, gate, out, out_stride, ks, s);
    return launch_portions<bf16>(q, kc, vc, positions, seq_idx, block_tables, bt_stride, T, H, G, dk, dv, ldv, pitch, scale,
                                 gate, out, out_stride, ks, s);
}
