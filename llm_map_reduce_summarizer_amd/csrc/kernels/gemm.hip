// Large-M fp8 GEMM on the matrix cores (prefill projections of 8-bit models), and the entry point of both tile GEMMs:
//
//     C[M, N] = X[M, K] . W[N, K]^T            X = activations, W = weights, both K-contiguous
//
//   * bf16 x bf16 runs in gemm_bf16.hip;
//   * OCP e4m3fn x e4m3fn on v_mfma_scale_f32_16x16x128_f8f6f4 with unit block scales (E8M0 127): the
//     block-scaled form runs at twice the bf16 rate (MI355X_MICROARCH.md "Matrix cores"), so the plain
//     per-row quantisation (activation row scale sx[m] x weight row scale sw[n]) is applied in the
//     epilogue and the MX block scales stay 1.0.  (Per-32 E8M0 activation scales measured WORSE than the
//     fp32 row scale: power-of-two scales waste up to a bit of e4m3's range -- 2.67 vs 2.29 % element
//     error, 25.6 vs 24.3 % on the fp8 parity logits, profiles/r4_fp8_activation_emulation.txt.)
//   * two-term fp8 activations (norm.hip Q8 == 2, the fp8 model's QKV input): X rows hold [hi | lo] over
//     2K bytes, W keeps K; the K-tiles kt >= kbw (the lo half) re-read W's tile kt - kbw and run with the
//     X block scale E8M0 123 = 2^-4, so one launch computes hi W^T + lo W^T / 16.
//
// Structure (cdna_hip_programming.md §5 "The 256^2 8-phase template", re-derived for this layout):
//   * one 256 x 256 output tile per 512-thread workgroup (8 waves, one workgroup per CU), K-tiles of 128
//     bytes per row (128 e4m3); the XCD-aware bijective tile remap + grouped raster keeps
//     the ~32 tiles an XCD runs at a time on 4 X row-panels x 8 W row-panels (L2 reuse).
//   * LDS: 2 buffers x 4 half-tile images of 128 rows x 128 B (X rows 0-127, W rows 0-127, W rows
//     128-255, X rows 128-255 -- the order the phases first read them) = 128 KiB in ONE __shared__
//     array.  Half-tiles arrive by LDS-DMA (buffer_load ... lds, 16 B per lane, one 1 KiB piece = 8
//     rows per wave instruction) from a tile-local buffer descriptor: rows past M / N are dropped by
//     the descriptor's range check (their LDS rows hold stale bytes that only feed masked outputs).
//     The bank swizzle is applied on the SOURCE address (rule 21): 16-B chunk c of row r sits at
//     chunk position c ^ ((r >> 1) & 7), which makes every ds_read_b128 fragment read conflict-free
//     (each 16-lane group covers the 16 slots of a bank row).
//   * wave (wr, wc) owns 128 x 64 outputs split into four 64 x 32 quadrants; quadrant (qm, qn) reads
//     X half qm and W half qn, so the four phases of a K-tile need the half-tiles in the order
//     X0 W0 | W1 | X1 | -- and a half-tile can be staged LOOK = 6 half-tiles (1.5 K-tiles) ahead of
//     the phase that first reads it.  Per phase: R = fragment ds_reads + stage one half-tile (2 DMA
//     per lane) + counted s_waitcnt vmcnt(8) (never 0 in the main loop), raw s_barrier, M = 8
//     MFMAs between s_setprio(1/0), raw s_barrier.  Waves 4-7 run one barrier (half a phase)
//     behind waves 0-3 (stagger), so one wave of each SIMD reads LDS while its partner computes.
//   * hazards (derived for the staggered schedule, which is the stricter one): the wait at the end of
//     R_P covers every half-tile phase P+1 reads, before the barrier the lagging group passes ahead
//     of its R_P; a half-tile is restaged >= 2 phases after the last phase that read its region
//     (reads are retired by the lgkmcnt wait ahead of that phase's MFMAs, which precede the barrier
//     the restaging wave passes).
//   * the MFMA computes the transposed tile (A = W fragment, B = X fragment) so each lane ends with 4
//     consecutive output columns of one row: 8-byte bf16 stores, and the fused SwiGLU epilogue of the
//     [8 gate | 8 up]-interleaved gate_up weight is a lane-xor-32 exchange.
//   * split tail: as in gemm_bf16.hip, with this kernel's register order.
//   * M32 variant: the same ring, phases and quadrants on 32x32 MFMA tiles
//     (v_mfma_scale_f32_32x32x64_f8f6f4); a lane then holds 4 register groups of 4 consecutive columns,
//     and the SwiGLU gate / up halves of a 16-column group sit in adjacent groups of the same lane.
#include "gemm.h"

#include <type_traits>

namespace {
constexpr int HALF = 16384;
constexpr int TILE = 4 * HALF;
constexpr int LOOK = 6;

typedef int i32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void vm_wait_rt(int n) {
    if (n >= 12) vm_wait<12>();
    else if (n >= 10) vm_wait<10>();
    else if (n >= 8) vm_wait<8>();
    else if (n >= 6) vm_wait<6>();
    else if (n >= 4) vm_wait<4>();
    else if (n >= 2) vm_wait<2>();
    else vm_wait<0>();
}

__device__ __forceinline__ void bar() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
}  // namespace

template <int EPI, int NS, bool LEPI, bool M32>
__global__ __launch_bounds__(512, 1) void gemm_kernel(const GemmArgs a) {
    // NS = half-tile slots of the LDS ring: half-tile h (K-tile h / 4, part h % 4) lives in slot h % NS.
    // NS = 8 (128 KiB, 2 K-tiles): staged LK = 6 ahead; NS = 10 (160 KiB): LK = 8 ahead.  A slot is
    // restaged at phase h + NS - LK >= 2 phases after the last phase that read half-tile h (<= h).
    constexpr int LK = NS - 2;
    static_assert(NS * HALF <= 160 * 1024 && NS * HALF >= 2 * TILE, "LDS ring size");
    __shared__ __attribute__((aligned(1024))) char lds[NS * HALF];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w >> 2, wc = w & 3;
    int tm, tn;
    // whole tiles first; then the slices, one K range after the other, so that an XCD's slices read the same panels
    int pos, slice = -1, kt0 = 0, kt1 = a.kb;
    if ((int)blockIdx.x < a.whole) {
        pos = xcd_position(blockIdx.x, a.whole);
    } else {
        const int rest = a.tiles_m * a.tiles_n - a.whole;
        const int p = xcd_position(blockIdx.x - a.whole, gridDim.x - a.whole);
        slice = p / rest;
        pos = a.whole + p - slice * rest;
        kt0 = a.kb * slice / a.splits;
        kt1 = a.kb * (slice + 1) / a.splits;
    }
    tile_of(pos, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
    const int m0 = tm * 256, n0 = tn * 256;
    const int xrows = min(a.M - m0, 256), wrows = min(a.N - n0, 256);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + (size_t)m0 * a.ldx_b), (short)0, xrows * a.ldx_b, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.w + (size_t)n0 * a.ldw_b), (short)0, wrows * a.ldw_b, 0x00020000);

    // staging: this lane's source offsets for the 2 pieces (8 rows each) of every half-tile it fills
    const int srow = 16 * w + (lane >> 3);
    const int ch0 = ((lane & 7) ^ ((lane >> 4) & 7)) << 4;
    const int ch1 = ((lane & 7) ^ ((4 + (lane >> 4)) & 7)) << 4;
    const int vx0 = srow * a.ldx_b + ch0, vx1 = (srow + 8) * a.ldx_b + ch1;
    const int vw0 = srow * a.ldw_b + ch0, vw1 = (srow + 8) * a.ldw_b + ch1;
    const int xh = 128 * a.ldx_b, wh = 128 * a.ldw_b;
    const int nk = kt1 - kt0, htot = 4 * nk;

    auto stage = [&](int part, int kt) {
        char* dst = lds + ((4 * kt + part) % NS) * HALF + w * 2048;
        kt += kt0;
        const int soff = kt * 128;
        if (part == 0 || part == 3) {
            const int o = part == 3 ? xh : 0;
            dma16(rx, dst, vx0 + o, soff);
            dma16(rx, dst + 1024, vx1 + o, soff);
        } else {
            const int o = part == 2 ? wh : 0;
            const int sw = (kt >= a.kbw ? kt - a.kbw : kt) * 128;
            dma16(rw, dst, vw0 + o, sw);
            dma16(rw, dst + 1024, vw1 + o, sw);
        }
    };

    // fragment reads.  16x16 MFMA: row (lane & 15) of a 16-row block, chunk (lane >> 4) (k-step 0) or
    // 4 + (lane >> 4).  32x32 MFMA (M32): row (lane & 31) of a 32-row block, read r = chunk 2 r + (lane >> 5);
    // any k order shared by the A and B operands gives the same dot product, and each ds_read_b128 lane
    // group still covers 16 distinct slots of a bank row (rows r, r + 1 share the swizzle, 8 slots apart).
    int lo[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        lo[r] = M32 ? (lane & 31) * 128 + (((2 * r + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4)
                    : (lane & 15) * 128 + (((4 * (r & 1) + (lane >> 4)) ^ ((lane >> 1) & 7)) << 4);
    const int xbase = (64 * wr) * 128, wbase = (32 * wc) * 128;

    // per quadrant: 16x16 -- [x block b 0..3][w block i 0..1] f32x4; 32x32 -- [x block b 0..1] f32x16
    f32x4 acc[2][4][2][2];
    f32x16 acc32[2][2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    if constexpr (M32) { if (b < 2 && k == 0) acc32[i][b][j] = f32x16{}; }
                    else acc[i][b][j][k] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
    // xf[2 b + ks] (16x16) | xf[4 b + r] (32x32); wf[2 i + ks] | wf[r]
    u32x4 xf[8], wf0[4], wf1[4];

    // prologue: half-tiles 0 .. LK-1 in flight, wait for the phase 0 reads (h <= 1 | h <= 2)
#pragma unroll
    for (int h = 0; h < LK; ++h)
        if (h < htot) stage(h & 3, h >> 2);
    vm_wait_rt(2 * (min(LK - 1, htot - 1) - 1));
    bar();
    if (wr == 1) bar();  // stagger: waves 4-7 run one barrier (half a phase) behind waves 0-3

    // 16x16: block b (16 rows) read ks at b * 2048 + lo[ks];  32x32: block b (32 rows) read r at b * 4096 + lo[r]
    auto read_x = [&](const char* base) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xf[j] = *reinterpret_cast<const u32x4*>(base + xbase + (M32 ? (j >> 2) * 4096 + lo[j & 3]
                                                                        : (j >> 1) * 2048 + lo[j & 1]));
    };
    auto read_w = [&](const char* base, u32x4 (&wf)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            wf[j] = *reinterpret_cast<const u32x4*>(base + wbase + (M32 ? lo[j] : (j >> 1) * 2048 + lo[j & 1]));
    };
    auto cat8 = [](const u32x4& p, const u32x4& q) -> i32x8 {
        return i32x8{(int)p[0], (int)p[1], (int)p[2], (int)p[3], (int)q[0], (int)q[1], (int)q[2], (int)q[3]};
    };
    auto mfma_q = [&](int qm, int qn, const u32x4 (&wf)[4], int xsc) {
        __builtin_amdgcn_s_setprio(1);
        if constexpr (M32) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    acc32[qm][b][qn] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                        cat8(wf[2 * s], wf[2 * s + 1]), cat8(xf[4 * b + 2 * s], xf[4 * b + 2 * s + 1]),
                        acc32[qm][b][qn], 0, 0, 0, 127, 0, xsc);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc[qm][b][qn][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        cat8(wf[2 * i], wf[2 * i + 1]), cat8(xf[2 * b], xf[2 * b + 1]), acc[qm][b][qn][i], 0, 0, 0,
                        127, 0, xsc);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // stage the half-tile LK ahead of phase P = 4 kt + p, then wait for what phase P + 1 reads.  In the
    // steady state (TAIL false: kt < nk - LK / 4) the stage always exists and the wait is vmcnt(2 (LK - 2)).
    auto stage_and_wait = [&](int kt, int p, auto tail) {
        const int P = 4 * kt + p, h = P + LK;
        if constexpr (decltype(tail)::value) {
            if (h < htot) stage(h & 3, h >> 2);
            const int rem = htot - 1 - P;
            vm_wait_rt(rem >= LK ? 2 * (LK - 2) : 2 * (rem - 2));
        } else {
            stage(h & 3, h >> 2);
            vm_wait<2 * (LK - 2)>();
        }
    };
    auto slot = [&](int kt, int part) -> const char* { return lds + ((4 * kt + part) % NS) * HALF; };
    auto ktile = [&](int kt, auto tail) {
        const int xsc = kt0 + kt >= a.kbw ? 123 : 127;  // E8M0 2^-4 on the lo half of two-term X
        // phase 0: quadrant (0, 0) -- X0, W0
        read_x(slot(kt, 0));
        read_w(slot(kt, 1), wf0);
        stage_and_wait(kt, 0, tail);
        bar();
        mfma_q(0, 0, wf0, xsc);
        bar();
        // phase 1: quadrant (0, 1) -- W1
        read_w(slot(kt, 2), wf1);
        stage_and_wait(kt, 1, tail);
        bar();
        mfma_q(0, 1, wf1, xsc);
        bar();
        // phase 2: quadrant (1, 1) -- X1
        read_x(slot(kt, 3));
        stage_and_wait(kt, 2, tail);
        bar();
        mfma_q(1, 1, wf1, xsc);
        bar();
        // phase 3: quadrant (1, 0) -- registers only
        stage_and_wait(kt, 3, tail);
        bar();
        mfma_q(1, 0, wf0, xsc);
        bar();
    };
    // steady state while every phase's stage exists: P + LK < htot for P <= 4 kt + 3
    int kt = 0;
    for (; kt < nk - (LK + 3) / 4; ++kt) ktile(kt, std::false_type{});
    for (; kt < nk; ++kt) ktile(kt, std::true_type{});
    if (wr == 0) bar();

    if constexpr (!M32) {
        if (slice >= 0) {
            // accumulator vector v of this lane at [v][thread]; 16-row blocks past M are skipped
            f32x4* out = reinterpret_cast<f32x4*>(a.part + ((size_t)(pos - a.whole) * a.splits + slice) * TILE_F) + tid;
#pragma unroll
            for (int qm = 0; qm < 2; ++qm)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (128 * qm + 64 * wr + 16 * b >= xrows) continue;
#pragma unroll
                    for (int v = 0; v < 4; ++v) out[((qm * 4 + b) * 4 + v) * 512] = acc[qm][b][v >> 1][v & 1];
                }
            return;
        }
    }

    // epilogue: lane holds C[m][n .. n+3] of every 16 x 16 block, m = .. + (lane & 15), n = .. + 4 (lane >> 4).
    // LEPI: every wave writes its bf16 results into a [256 rows][RB bytes] LDS image of the whole tile
    // (16-B unit u of row r at u ^ (r & 7): 2-way ds_write_b64, conflict-free ds_read_b128), then each
    // wave stores 32 whole rows with 16-B lanes (full-row segments instead of 32-B pieces per row).
    constexpr int RB = EPI == GEPI_SWIGLU ? 256 : 512;
    // fp8: v *= activation row scale x weight row scales of tile columns c4 .. c4+3
    auto scale4 = [&](f32x4& v, float rs, int c4) {
        const float4 s4 = *reinterpret_cast<const float4*>(a.sw + min(n0 + c4, a.N - 4));
        v[0] *= rs * s4.x; v[1] *= rs * s4.y; v[2] *= rs * s4.z; v[3] *= rs * s4.w;
    };
    auto silu_mul = [&](const f32x4& g, const f32x4& u) {
        f32x4 r;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = glu(g[j], u[j], a.glu);
        return r;
    };
    // 4 bf16 outputs of tile row rl at byte cbyte of the output tile row; gcol = first weight column of
    // the 16-column group they come from (N % 16 == 0, so the group is wholly in or out of range)
    auto store4 = [&](int rl, int cbyte, f32x4 v, int gcol) {
        const uint2 pk = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
        if constexpr (LEPI) {
            *reinterpret_cast<uint2*>(lds + rl * RB + (((cbyte >> 4) ^ (rl & 7)) << 4) + (cbyte & 15)) = pk;
        } else if (m0 + rl < a.M && n0 + gcol < a.N) {
            char* o = reinterpret_cast<char*>(a.c) + ((size_t)(m0 + rl) * a.ldc) * 2 +
                      (EPI == GEPI_SWIGLU ? n0 : 2 * n0) + cbyte;
            *reinterpret_cast<uint2*>(o) = pk;
        }
    };
    if constexpr (M32) {
        // lane holds C[m][n .. n+3] of every 32 x 32 block: m = .. + (lane & 31), register group gi covers
        // n = .. + 8 gi + 4 (lane >> 5).  SwiGLU: groups 0 / 2 are gate, 1 / 3 the matching up columns.
        const int h = lane >> 5;
#pragma unroll
        for (int qm = 0; qm < 2; ++qm)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int rl = 128 * qm + 64 * wr + 32 * b + (lane & 31);
                const float rs = a.sx[min(m0 + rl, a.M - 1)];
#pragma unroll
                for (int qn = 0; qn < 2; ++qn) {
                    const int cb = 128 * qn + 32 * wc;
                    f32x4 v[4];
#pragma unroll
                    for (int gi = 0; gi < 4; ++gi) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) v[gi][t] = acc32[qm][b][qn][4 * gi + t];
                        scale4(v[gi], rs, cb + 8 * gi + 4 * h);
                    }
                    if constexpr (EPI == GEPI_SWIGLU) {
#pragma unroll
                        for (int gp = 0; gp < 2; ++gp) {
                            const int gcol = cb + 16 * gp;
                            store4(rl, ((gcol >> 1) + 4 * h) * 2, silu_mul(v[2 * gp], v[2 * gp + 1]), gcol);
                        }
                    } else {
#pragma unroll
                        for (int gi = 0; gi < 4; ++gi) {
                            const int c4 = cb + 8 * gi + 4 * h;
                            store4(rl, c4 * 2, v[gi], c4);
                        }
                    }
                }
            }
    } else {
        // lane holds C[m][n .. n+3] of every 16 x 16 block, m = .. + (lane & 15), n = .. + 4 (lane >> 4).
        // SwiGLU: the up columns 8-15 of a 16-column group sit in lane xor 32.
        const int g4 = lane >> 4;
#pragma unroll
        for (int qm = 0; qm < 2; ++qm)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int rl = 128 * qm + 64 * wr + 16 * b + (lane & 15);
                const float rs = a.sx[min(m0 + rl, a.M - 1)];
#pragma unroll
                for (int qn = 0; qn < 2; ++qn)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const int cb = 128 * qn + 32 * wc + 16 * i;  // 16-column block within the tile
                        f32x4 v = acc[qm][b][qn][i];
                        scale4(v, rs, cb + 4 * g4);
                        if constexpr (EPI == GEPI_SWIGLU) {
                            f32x4 up;
#pragma unroll
                            for (int j = 0; j < 4; ++j) up[j] = __shfl_xor(v[j], 32, 64);
                            if (g4 < 2) store4(rl, ((cb >> 1) + 4 * g4) * 2, silu_mul(v, up), cb);
                        } else {
                            store4(rl, (cb + 4 * g4) * 2, v, cb);
                        }
                    }
            }
    }
    if constexpr (LEPI) {
        __syncthreads();
        constexpr int UPR = RB / 16, RPI = 1024 / RB;
#pragma unroll
        for (int it = 0; it < 32 / RPI; ++it) {
            const int rl = 32 * w + RPI * it + lane / UPR, u = lane % UPR;
            const u32x4 val = *reinterpret_cast<const u32x4*>(lds + rl * RB + ((u ^ (rl & 7)) << 4));
            const int m = m0 + rl;
            const int col = (EPI == GEPI_SWIGLU ? (n0 >> 1) : n0) + 8 * u;  // output column of the unit
            const bool ok = m < a.M && (EPI == GEPI_SWIGLU ? 2 * col : col) < a.N;
            if (ok) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(a.c) + (size_t)m * a.ldc + col) = val;
        }
    }
}

// Adds the slices of the split tiles and runs the epilogue.  One workgroup per (tile, 2 x 16 rows): the four vectors
// that every lane of gemm_kernel holds for one of its eight row blocks.
template <int EPI>
__global__ __launch_bounds__(512) void gemm_tail_kernel(const GemmArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 2, wc = w & 3, g4 = lane >> 4;
    const int t = blockIdx.x >> 3, rb = blockIdx.x & 7;
    int tm, tn;
    tile_of(a.whole + t, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
    const int n0 = tn * 256, r0 = tm * 256 + 128 * (rb >> 2) + 64 * wr + 16 * (rb & 3);
    if (r0 >= a.M) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * TILE_F) + rb * 4 * 512 + tid;
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = in[j * 512];
    for (int s = 1; s < a.splits; ++s) {
        in += TILE_F / 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += in[j * 512];
    }
    const int m = r0 + (lane & 15);
    const float rs = a.sx[min(m, a.M - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int cb = n0 + 128 * (j >> 1) + 32 * wc + 16 * (j & 1);  // 16-column block, wholly in or out of range
        const float4 s4 = *reinterpret_cast<const float4*>(a.sw + min(cb + 4 * g4, a.N - 4));
        v[j][0] *= rs * s4.x; v[j][1] *= rs * s4.y; v[j][2] *= rs * s4.z; v[j][3] *= rs * s4.w;
        int col = cb + 4 * g4;
        if constexpr (EPI == GEPI_SWIGLU) {  // the up columns sit in lane xor 32
            f32x4 up;
#pragma unroll
            for (int k = 0; k < 4; ++k) up[k] = __shfl_xor(v[j][k], 32, 64);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[j][k] = glu(v[j][k], up[k], a.glu);
            col = (cb >> 1) + 4 * g4;
        }
        if (m >= a.M || cb >= a.N || (EPI == GEPI_SWIGLU && lane >= 32)) continue;
        *reinterpret_cast<uint2*>(reinterpret_cast<bf16*>(a.c) + (size_t)m * a.ldc + col) =
            make_uint2(pack2(v[j][0], v[j][1]), pack2(v[j][2], v[j][3]));
    }
}

#ifdef MRSUM_CLOCK_STAMPS
static unsigned long long* g_stamps = nullptr;
static int g_nstamps = 0;
// copies the last launch's [grid][2] stamps to host memory; returns the count of u64 words (diagnostic build)
MRSUM_API int mrsum_gemm_stamps(unsigned long long* host, int max_words) {
    const int n = std::min(max_words, g_nstamps);
    if (!g_stamps || n <= 0 || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(host, g_stamps, (size_t)n * 8, hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    return n;
}
#endif

// x [M, K] (row stride ldx elements), w [N, K] (ldw), c [M, N] bf16 (ldc) -- or [M, N / 2] for
// epi 1 (SwiGLU of the [8 gate | 8 up]-interleaved gate_up rows) -- or gelu(C) for epi 2, or C in
// fp32 for epi 3 (both bf16 operands only).  fp8: x, w are e4m3fn bytes,
// sx [M] / sw [N] fp32 row scales; split: x is two-term [hi | lo] of 2K bytes per row over w's K.
// whole / splits / part: tiles from raster position ``whole`` on run in ``splits`` slices of K through ``part``
// [tiles - whole][splits][rows * 256] fp32 (splits 1: none, part unused;
// 16x16 MFMA tiles only).  group_m bits 9 - 12: rows of a tile / 32 (0: 256; bf16 also 128, 160, 192, 224).  slabs (epi 3,
// whole 0): the slices stay apart, in part [splits][M][N]; c unused.
// Requirements (checked by the Python wrapper too): K % 64 and K > 0 (bf16) / K % 128 (fp8), N % 16, 16-byte
// aligned rows.
MRSUM_API int mrsum_gemm(const void* x, int ldx, const void* w, int ldw, void* c, int ldc, int M, int N, int K,
                         int fp8, int epi, const float* sx, const float* sw, int group_m, int split, float glu_limit,
                         float glu_alpha, float glu_shift, int whole, int splits, float* part, int slabs,
                         hipStream_t s) {
    if (M <= 0 || N <= 0) return 0;
    const int es = fp8 ? 1 : 2;
    if ((K * es) % 128 || N % 16 || (ldx * es) % 16 || (ldw * es) % 16 || ldc % 4) return (int)hipErrorInvalidValue;
    if ((size_t)256 * ldx * es >= (1u << 31) || (size_t)256 * ldw * es >= (1u << 31)) return (int)hipErrorInvalidValue;
    if (epi < GEPI_BF16 || epi > GEPI_F32 || (epi >= GEPI_GELU && (fp8 || ((group_m >> 8) & 1))))
        return (int)hipErrorInvalidValue;
    if (fp8 ? !sx || !sw : K < 64) return (int)hipErrorInvalidValue;
    const int rows = (group_m >> 9) & 15 ? 32 * ((group_m >> 9) & 15) : 256;
    if (rows != 256 && (fp8 || rows < 128 || rows > 256)) return (int)hipErrorInvalidValue;
    GemmArgs a;
    a.x = (const char*)x; a.w = (const char*)w; a.c = c; a.sx = sx; a.sw = sw;
    a.ldx_b = ldx * es; a.ldw_b = ldw * es; a.ldc = ldc;
    a.M = M; a.N = N; a.kb = K * es / 128;
    a.glu = GluArgs{glu_limit, glu_alpha, glu_shift};
    if (split && (!fp8 || ldx < 2 * K)) return (int)hipErrorInvalidValue;
    a.kbw = a.kb;
    if (split) a.kb *= 2;  // X K-tiles: hi then lo
    a.rows = rows;
    a.tiles_m = ceil_div(M, rows); a.tiles_n = ceil_div(N, 256);
    // group_m bits 0-7: tile rows per raster group (0 = 4); bit 8: fp8 on 32x32 MFMA tiles instead of 16x16 (bf16 has one form).
    // Measured (profiles/r3_gemm_mfma32_experiment.jsonl, same box, interleaved): 32x32 is
    // about equal on the 70B fp8 qkv / o / down, so 16x16 stays the default;
    // the gate_up + SwiGLU GEMM gains 1.7-3.8 % at M = 4k-32k and takes it (ops/hip.py gemm_fp8).
    const bool m32 = fp8 && ((group_m >> 8) & 1);
    group_m &= 255;
    a.group_m = group_m > 0 ? group_m : 4;
    const int tiles = a.tiles_m * a.tiles_n;
    if (splits > 1 && (whole < 0 || whole >= tiles || splits > a.kb || !part || m32))
        return (int)hipErrorInvalidValue;
    a.splits = splits > 1 ? splits : 1;
    a.whole = splits > 1 ? whole : tiles;
    a.part = part;
    a.slabs = slabs;
    if (slabs && (epi != GEPI_F32 || splits <= 1 || whole || N % 16)) return (int)hipErrorInvalidValue;
    const int rest = tiles - a.whole;
    if (!fp8) {
#ifdef MRSUM_CLOCK_STAMPS
        const size_t wgs = gemm_bf16_grid(a);
        static unsigned long long* stamps = nullptr;
        static size_t nstamps = 0;
        if (nstamps < 2 * wgs) {
            if (stamps) (void)hipFree(stamps);
            nstamps = 2 * wgs;
            if (hipMalloc(&stamps, nstamps * 8) != hipSuccess) return (int)hipErrorOutOfMemory;
        }
        a.stamps = stamps;
        g_stamps = stamps;
        g_nstamps = 2 * (int)wgs;
#endif
        gemm_bf16_launch(a, epi, s);
        return (int)hipGetLastError();
    }
    const dim3 grid(a.whole + rest * a.splits), block(512);
    // measured (profiles/r2_gemm_variants_ab.jsonl, r2_gemm_ring10_ab.jsonl): the staggered 8-slot ring
    // (LOOK 6) with the LDS-staged epilogue is the fastest; the 2-phase / 10-slot rings and the
    // unstaggered schedule lost 5-25 %.  The register epilogue remains for outputs that are not 16-B
    // aligned (strided views).
    const bool lepi = ldc % 8 == 0 && (uintptr_t)c % 16 == 0;
#define GEMM_LAUNCH(E)                                                          \
    if (m32) {                                                                  \
        if (lepi) gemm_kernel<E, 8, true, true><<<grid, block, 0, s>>>(a);      \
        else gemm_kernel<E, 8, false, true><<<grid, block, 0, s>>>(a);          \
    } else {                                                                    \
        if (lepi) gemm_kernel<E, 8, true, false><<<grid, block, 0, s>>>(a);     \
        else gemm_kernel<E, 8, false, false><<<grid, block, 0, s>>>(a);         \
        if (rest) gemm_tail_kernel<E><<<rest * 8, block, 0, s>>>(a);            \
    }
    if (epi == GEPI_SWIGLU) { GEMM_LAUNCH(GEPI_SWIGLU) } else { GEMM_LAUNCH(GEPI_BF16) }
#undef GEMM_LAUNCH
    return (int)hipGetLastError();
}
