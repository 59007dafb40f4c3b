// Large-M bf16 GEMM (prefill projections, LM head over many rows):
//
//     C[M, N] = X[M, K] . W[N, K]^T            X = activations, W = weights, both K-contiguous
//
// One 256 x 256 output tile at a time per workgroup of four waves, one wave per SIMD; wave (wr, wc) owns 128 x 128 outputs
// = 8 x 8 blocks of v_mfma_f32_16x16x32_bf16 in all 256 accumulation registers.  What bounds it: LDS and the matrix
// cores.  A K-tile of 64 is 2048 cycles of MFMA per SIMD; eight waves of 128 x 64 read 192 KiB of fragments for it and fill
// 64 KiB by DMA, which is as many LDS cycles again, and took 2760 - 2850; four waves read 128 KiB and take 2200.
// What else the fewer waves need is that nothing but the matrix cores is ever waited for, as no second wave covers a
// SIMD's waits, so the loop over K is written out:
//
//   * LDS: a ring of five 32 KiB images of 256 rows x 128 B (160 KiB), X and W K-tiles in turn (X0 W0 X1 W1 X2 | W2 ...).
//     Images arrive by LDS-DMA (buffer_load ... lds, 1 KiB = 8 rows per wave instruction) from a tile-local buffer
//     descriptor: rows past M / N are dropped by the descriptor's range check (their LDS rows hold stale bytes that
//     only feed masked outputs).  The bank swizzle is on the SOURCE address: 16-byte chunk c of row r sits at position
//     c ^ f(r), f taking all eight values over the rows that one fragment read touches.
//   * K-tile t: step 0 runs the 64 MFMAs of k 0 - 31 while the fragments of k 32 - 63 come from LDS into the other
//     register set and X(t + 2) is requested; then the one wait and barrier of the K-tile: every wave has its fragments
//     of t, and X, W(t + 1) have arrived; step 1 runs k 32 - 63 while the first fragments of t + 1 are read and W(t + 2)
//     is requested into the image that X(t) leaves.
//   * the workgroups stay for all their tiles, and the requests run on into the next tile (or slice of K), whose first two
//     K-tiles arrive while the epilogue runs.  The epilogue keeps out of LDS for that: W's rows are dealt to the MFMA
//     rows so that a lane ends with 8 consecutive output columns (gate and up of the same columns for GLU) of a row, one
//     16-byte store, 64 bytes in a row by four lanes.
//   * the MFMA computes the transposed tile (A = W fragment, B = X fragment); column blocks go back and forth over the row
//     blocks, so that a neighbour's operand stays.
//   * split tail: tiles behind the last whole round of 256 (all of them where M and N are small) would leave most CUs
//     idle for a full K loop, so each is cut into S slices of K.  A slice writes its fp32 accumulators to scratch in
//     register order (lane-contiguous 16-B stores) and gemm_bf16_tail_kernel adds them in slice order and runs the
//     epilogue: a second launch and no ticket, so results do not depend on arrival and concurrent streams share
//     nothing.  Which S: ops/hip.py gemm_splits.
//
// Measured, eight waves (two 64 KiB tiles of LDS, two barriers a quarter of a K-tile) -> this, us: 18234 x 28672 x 4096 with
// GLU 3498 -> 3051 (1404 TFLOP/s), 18234 x 4096 x 14336 1592 -> 1441 (1486), 18234 x 6144 x 4096 694 -> 654, 4096 x 4096 x
// 22528 549 -> 507, 1967 x 24576 x 4096 with gelu 322 -> 292, 300 x 4096 x 14336 in slices 54.4 -> 50.5.  The large ones run
// at the clock that the card's power allows (1.7 - 1.9 of 2.4 GHz), so fewer cycles only partly show as time.
#include "gemm.h"

namespace {
constexpr int IMAGE = 256 * 128;  // one operand's K-tile
constexpr int RING = 5 * IMAGE;
constexpr int WGS = 256;          // one workgroup per CU

// ---- the loop over K as text.  Fragment set s: X blocks in v[128 + 64 s ..], W blocks in v[160 + 64 s ..]; accumulators
// of (W block j, X block b) in a[32 j + 4 b ..]; descriptors of X and W in s[64:67] and s[68:71], of what follows this
// unit in s[72:75] and s[76:79].
#define STR_(...) #__VA_ARGS__
#define STR(...) STR_(__VA_ARGS__)
#define XF(s, b) "v[" STR(128 + 64 * s + 4 * b) ":" STR(131 + 64 * s + 4 * b) "]"
#define WF(s, j) "v[" STR(160 + 64 * s + 4 * j) ":" STR(163 + 64 * s + 4 * j) "]"
#define ACC(j, b) "a[" STR(32 * j + 4 * b) ":" STR(32 * j + 4 * b + 3) "]"
#define MF(s, j, b) "v_mfma_f32_16x16x32_bf16 " ACC(j, b) ", " WF(s, j) ", " XF(s, b) ", " ACC(j, b) "\n"
#define MZ(s, j, b) "v_mfma_f32_16x16x32_bf16 " ACC(j, b) ", " WF(s, j) ", " XF(s, b) ", 0\n"
// one row block against all column blocks, with room for three fragment reads and a request in between
#define ROW(M, s, b, r0, r1, r2, d)  M(s, 0, b) M(s, 1, b) r0 M(s, 2, b) M(s, 3, b) r1 M(s, 4, b) M(s, 5, b) r2 M(s, 6, b) M(s, 7, b) d
#define BACK(M, s, b, r0, r1, r2, d) M(s, 7, b) M(s, 6, b) r0 M(s, 5, b) M(s, 4, b) r1 M(s, 3, b) M(s, 2, b) r2 M(s, 1, b) M(s, 0, b) d
#define RX(s, b) "ds_read_b128 " XF(s, b) ", %[xa] offset:" STR(2048 * b) "\n"
#define RW(s, j, off) "ds_read_b128 " WF(s, j) ", %[wa] offset:" STR(128 * off(j)) "\n"
#define DX(p) "buffer_load_dwordx4 %[vx" #p "], s[64:67], %[kd] offen lds\ns_add_u32 m0, m0, 0x400\n"
#define DW(p) "buffer_load_dwordx4 %[vw" #p "], s[68:71], %[kd] offen lds\ns_add_u32 m0, m0, 0x400\n"
#define READ_AT(x, w) "v_add_u32 %[xa], %[sx], %[" x "]\nv_add_u32 %[wa], %[sw], %[" w "]\n"
#define NEXT_SLOT(r) "s_add_u32 %[" r "], %[" r "], 0x10000\ns_cmp_ge_u32 %[" r "], 0x28000\n" \
                     "s_cselect_b32 %[t0], 0x28000, 0\ns_sub_u32 %[" r "], %[" r "], %[t0]\n"
#define STEP0(M, off)                                                                       \
    READ_AT("xlo1", "wlo1") "s_add_u32 m0, %[sp], %[ldsw]\n"                                \
    ROW(M, 0, 0, RX(1, 0), RX(1, 1), RX(1, 2), DX(0))                                       \
    BACK(M, 0, 1, RX(1, 3), RX(1, 4), RX(1, 5), DX(1))                                      \
    ROW(M, 0, 2, RX(1, 6), RX(1, 7), RW(1, 0, off), DX(2))                                  \
    BACK(M, 0, 3, RW(1, 1, off), RW(1, 2, off), RW(1, 3, off), DX(3))                       \
    ROW(M, 0, 4, RW(1, 4, off), RW(1, 5, off), , DX(4))                                     \
    BACK(M, 0, 5, RW(1, 6, off), RW(1, 7, off), , DX(5))                                    \
    ROW(M, 0, 6, , , , DX(6))                                                               \
    BACK(M, 0, 7, , , , DX(7))
#define STEP1(off)                                                                          \
    READ_AT("xlo0", "wlo0") "s_add_u32 m0, %[tp], %[ldsw]\n"                                \
    ROW(MF, 1, 0, RX(0, 0), RX(0, 1), RX(0, 2), DW(0))                                      \
    BACK(MF, 1, 1, RX(0, 3), RX(0, 4), RX(0, 5), DW(1))                                     \
    ROW(MF, 1, 2, RX(0, 6), RX(0, 7), RW(0, 0, off), DW(2))                                 \
    BACK(MF, 1, 3, RW(0, 1, off), RW(0, 2, off), RW(0, 3, off), DW(3))                      \
    ROW(MF, 1, 4, RW(0, 4, off), RW(0, 5, off), , DW(4))                                    \
    BACK(MF, 1, 5, RW(0, 6, off), RW(0, 7, off), , DW(5))                                   \
    ROW(MF, 1, 6, , , , DW(6))                                                              \
    BACK(MF, 1, 7, , , , DW(7))
// the requests have passed this unit's last K-tile: on to the next unit's first
#define FOLLOW                                                                              \
    "s_cmp_lg_u32 %[kd], %[ke]\ns_cbranch_scc1 3f\n"                                        \
    "s_mov_b64 s[64:65], s[72:73]\ns_mov_b64 s[66:67], s[74:75]\n"                          \
    "s_mov_b64 s[68:69], s[76:77]\ns_mov_b64 s[70:71], s[78:79]\n"                          \
    "s_mov_b32 %[kd], %[k0n]\ns_mov_b32 %[ke], %[ken]\n3:\n"
#define K_LOOP(off)                                                                         \
    "s_barrier\n" READ_AT("xlo0", "wlo0")                                                   \
    RX(0, 0) RX(0, 1) RX(0, 2) RX(0, 3) RX(0, 4) RX(0, 5) RX(0, 6) RX(0, 7)                 \
    RW(0, 0, off) RW(0, 1, off) RW(0, 2, off) RW(0, 3, off)                                 \
    RW(0, 4, off) RW(0, 5, off) RW(0, 6, off) RW(0, 7, off)                                 \
    FOLLOW "s_waitcnt lgkmcnt(0)\n" STEP0(MZ, off) "s_branch 2f\n"                          \
    "1:\n" FOLLOW "s_waitcnt lgkmcnt(0)\n" STEP0(MF, off)                                   \
    "2:\ns_waitcnt vmcnt(8) lgkmcnt(0)\ns_barrier\n"                                        \
    "s_mov_b32 %[tp], %[sx]\ns_mov_b32 %[sp], %[sw]\n" NEXT_SLOT("sx") NEXT_SLOT("sw")      \
    STEP1(off)                                                                              \
    "s_add_u32 %[kd], %[kd], 0x80\ns_sub_u32 %[n], %[n], 1\ns_cmp_lg_u32 %[n], 0\n"         \
    "s_cbranch_scc1 1b\ns_waitcnt lgkmcnt(0)\ns_nop 15\n"
// the W row of MFMA row a = lane & 15 of block j is OFF(j) + (8 or 16) (a >> 2) + (a & 3)
#define OFF_ROWS(j) (32 * (j >> 1) + 4 * (j & 1))
#define OFF_GLU(j) (64 * (j >> 2) + 4 * (j & 3))
#define ACC_OUTPUTS \
    "={a[0:3]}"(acc[0][0]), "={a[4:7]}"(acc[0][1]), "={a[8:11]}"(acc[0][2]), "={a[12:15]}"(acc[0][3]), \
    "={a[16:19]}"(acc[0][4]), "={a[20:23]}"(acc[0][5]), "={a[24:27]}"(acc[0][6]), "={a[28:31]}"(acc[0][7]), \
    "={a[32:35]}"(acc[1][0]), "={a[36:39]}"(acc[1][1]), "={a[40:43]}"(acc[1][2]), "={a[44:47]}"(acc[1][3]), \
    "={a[48:51]}"(acc[1][4]), "={a[52:55]}"(acc[1][5]), "={a[56:59]}"(acc[1][6]), "={a[60:63]}"(acc[1][7]), \
    "={a[64:67]}"(acc[2][0]), "={a[68:71]}"(acc[2][1]), "={a[72:75]}"(acc[2][2]), "={a[76:79]}"(acc[2][3]), \
    "={a[80:83]}"(acc[2][4]), "={a[84:87]}"(acc[2][5]), "={a[88:91]}"(acc[2][6]), "={a[92:95]}"(acc[2][7]), \
    "={a[96:99]}"(acc[3][0]), "={a[100:103]}"(acc[3][1]), "={a[104:107]}"(acc[3][2]), "={a[108:111]}"(acc[3][3]), \
    "={a[112:115]}"(acc[3][4]), "={a[116:119]}"(acc[3][5]), "={a[120:123]}"(acc[3][6]), "={a[124:127]}"(acc[3][7]), \
    "={a[128:131]}"(acc[4][0]), "={a[132:135]}"(acc[4][1]), "={a[136:139]}"(acc[4][2]), "={a[140:143]}"(acc[4][3]), \
    "={a[144:147]}"(acc[4][4]), "={a[148:151]}"(acc[4][5]), "={a[152:155]}"(acc[4][6]), "={a[156:159]}"(acc[4][7]), \
    "={a[160:163]}"(acc[5][0]), "={a[164:167]}"(acc[5][1]), "={a[168:171]}"(acc[5][2]), "={a[172:175]}"(acc[5][3]), \
    "={a[176:179]}"(acc[5][4]), "={a[180:183]}"(acc[5][5]), "={a[184:187]}"(acc[5][6]), "={a[188:191]}"(acc[5][7]), \
    "={a[192:195]}"(acc[6][0]), "={a[196:199]}"(acc[6][1]), "={a[200:203]}"(acc[6][2]), "={a[204:207]}"(acc[6][3]), \
    "={a[208:211]}"(acc[6][4]), "={a[212:215]}"(acc[6][5]), "={a[216:219]}"(acc[6][6]), "={a[220:223]}"(acc[6][7]), \
    "={a[224:227]}"(acc[7][0]), "={a[228:231]}"(acc[7][1]), "={a[232:235]}"(acc[7][2]), "={a[236:239]}"(acc[7][3]), \
    "={a[240:243]}"(acc[7][4]), "={a[244:247]}"(acc[7][5]), "={a[248:251]}"(acc[7][6]), "={a[252:255]}"(acc[7][7])
#define CLOBBER8(a) "v" #a "0", "v" #a "1", "v" #a "2", "v" #a "3", "v" #a "4", "v" #a "5", "v" #a "6", "v" #a "7", "v" #a "8", "v" #a "9"
#define CLOBBERS                                                                                                      \
    "memory", "scc", "m0", "v128", "v129", CLOBBER8(13), CLOBBER8(14), CLOBBER8(15), CLOBBER8(16), CLOBBER8(17),      \
        CLOBBER8(18), CLOBBER8(19), CLOBBER8(20), CLOBBER8(21), CLOBBER8(22), CLOBBER8(23), CLOBBER8(24), "v250",     \
        "v251", "v252", "v253", "v254", "v255"

__device__ __forceinline__ u32x4 descriptor(const char* p, int bytes) {
    const uint64_t v = (uint64_t)p;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)v),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) & 0xffff,
                 (uint32_t)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}

// One whole tile, or one slice of K of a tile.
struct Unit {
    int pos, slice, m0, n0, kt0, kt1;
};

__device__ __forceinline__ int units(const GemmArgs& a) {
    return a.whole + (a.tiles_m * a.tiles_n - a.whole) * a.splits;
}

// Whole tiles first, the 256 of a round spread over the XCDs; then the slices, one K range after the other, so that an
// XCD's slices read the same panels.
__device__ __forceinline__ Unit unit_of(const GemmArgs& a, int u) {
    Unit t;
    if (u < a.whole) {
        const int round = u & ~(WGS - 1);
        t.pos = round + xcd_position(u - round, min(a.whole - round, WGS));
        t.slice = -1;
        t.kt0 = 0;
        t.kt1 = a.kb;
    } else {
        const int rest = a.tiles_m * a.tiles_n - a.whole;
        const int p = xcd_position(u - a.whole, rest * a.splits);
        t.slice = p / rest;
        t.pos = a.whole + p - t.slice * rest;
        t.kt0 = a.kb * t.slice / a.splits;
        t.kt1 = a.kb * (t.slice + 1) / a.splits;
    }
    int tm, tn;
    tile_of(t.pos, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
    t.m0 = tm * 256;
    t.n0 = tn * 256;
    return t;
}

// Where a lane's outputs go: row block b is rows m0 + 16 b + (lane & 15); column group q (4, GLU 2) is 8 columns from col(q).
struct Lane {
    int m0, n0, wr, wc, r16, g4;
    __device__ __forceinline__ int row(int b) const { return 128 * wr + 16 * b + r16; }  // within the tile
};

// The outputs of column group q from a row block's accumulators v[j] (W block j).
template <int EPI>
__device__ __forceinline__ void outputs(const f32x4 (&v)[8], int q, const GluArgs& ga, float (&o)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        if constexpr (EPI == GEPI_SWIGLU) o[r] = glu(v[4 * q + (r >> 2)][r & 3], v[4 * q + 2 + (r >> 2)][r & 3], ga);
        else o[r] = v[2 * q + (r >> 2)][r & 3];
        if constexpr (EPI == GEPI_GELU) o[r] = gelu_tanh<bf16>(o[r]);
    }
}

// Row block b through the epilogue with stores of a form for any row length and alignment of 8 bytes (fp32: 16).
template <int EPI>
__device__ __forceinline__ void store_rows(const GemmArgs& a, const Lane& l, int b, const f32x4 (&v)[8]) {
    const int m = l.m0 + l.row(b);
    if (m >= a.M) return;
#pragma unroll
    for (int q = 0; q < (EPI == GEPI_SWIGLU ? 2 : 4); ++q) {
        const int n = l.n0 + 128 * l.wc + (EPI == GEPI_SWIGLU ? 64 * q + 16 * l.g4 : 32 * q + 8 * l.g4);
        if (n >= a.N) continue;
        if constexpr (EPI == GEPI_F32) {
            f32x4* o = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.c) + (size_t)m * a.ldc + n);
            o[0] = v[2 * q];
            o[1] = v[2 * q + 1];
        } else {
            float o[8];
            outputs<EPI>(v, q, a.glu, o);
            uint2* p = reinterpret_cast<uint2*>(reinterpret_cast<bf16*>(a.c) + (size_t)m * a.ldc + (EPI == GEPI_SWIGLU ? n >> 1 : n));
            p[0] = make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
            p[1] = make_uint2(pack2(o[4], o[5]), pack2(o[6], o[7]));
        }
    }
}
}  // namespace

// WIDE: rows of C are 16-byte aligned and 256 of them stay below 2 GiB, so that a whole tile leaves through a buffer
// descriptor in a fixed number of 16-byte stores, which the next tile's first wait can count past.
template <int EPI, bool WIDE>
__global__ __launch_bounds__(256, 1) void gemm_bf16_kernel(const GemmArgs a) {
    static_assert(!(WIDE && EPI == GEPI_F32), "fp32 rows leave by store_rows");
#ifdef MRSUM_CLOCK_STAMPS
    const unsigned long long clk0 = __builtin_amdgcn_s_memtime(), rt0 = __builtin_amdgcn_s_memrealtime();
#endif
    constexpr bool GLU = EPI == GEPI_SWIGLU;
    constexpr int STORES = GLU ? 16 : 32;
    __shared__ __attribute__((aligned(1024))) char lds[RING];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w >> 1, wc = w & 1;
    const int nu = units(a);

    // staging: wave w fills rows 64 w .. 64 w + 63 of an image in pieces of 8; position lane & 7 of row r takes chunk
    // (lane & 7) ^ f(r), f over bits 1 - 3 of an X row and the bits of a W row that a fragment read spans
    int vx[8], vw[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int r = 64 * w + 8 * p + (lane >> 3);
        const int fw = ((r >> 1) & 1) | (((r >> (GLU ? 4 : 3)) & 3) << 1);
        vx[p] = r * a.ldx_b + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
        vw[p] = r * a.ldw_b + (((lane & 7) ^ fw) << 4);
    }
    // fragment reads: row lane & 15 of a block, chunk lane >> 4 (step 0) or 4 + (lane >> 4) (step 1)
    const int fr = lane & 15, pos0 = ((lane >> 4) ^ (fr >> 1)) << 4;
    const int base = (int)(uintptr_t)(lds_ptr_t)lds;
    const int xlo0 = base + (128 * wr + fr) * 128 + pos0;
    const int wlo0 = base + (128 * wc + (GLU ? 16 : 8) * (fr >> 2) + (fr & 3)) * 128 + pos0;
    const int xlo1 = xlo0 ^ 64, wlo1 = wlo0 ^ 64, ldsw = base + w * 8192;

    Unit t = unit_of(a, blockIdx.x);
    u32x4 rx = descriptor(a.x + (size_t)t.m0 * a.ldx_b, min(a.M - t.m0, 256) * a.ldx_b);
    u32x4 rw = descriptor(a.w + (size_t)t.n0 * a.ldw_b, min(a.N - t.n0, 256) * a.ldw_b);
    {  // the first unit's first two K-tiles; a single one twice
        const __amdgpu_buffer_rsrc_t bx = rsrc(a.x + (size_t)t.m0 * a.ldx_b, min(a.M - t.m0, 256) * a.ldx_b);
        const __amdgpu_buffer_rsrc_t bw = rsrc(a.w + (size_t)t.n0 * a.ldw_b, min(a.N - t.n0, 256) * a.ldw_b);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int k = min(t.kt0 + i, t.kt1 - 1) * 128;
#pragma unroll
            for (int p = 0; p < 8; ++p) dma16(bx, lds + 2 * i * IMAGE + w * 8192 + p * 1024, vx[p], k);
#pragma unroll
            for (int p = 0; p < 8; ++p) dma16(bw, lds + (2 * i + 1) * IMAGE + w * 8192 + p * 1024, vw[p], k);
        }
    }
    vm_wait<16>();
    int sx = 0, sw = IMAGE, sp = 4 * IMAGE;  // images of X(t) and W(t), and the free one

    for (int u = blockIdx.x;;) {
        // what follows: the next unit, or a descriptor that drops every request
        const int un = u + gridDim.x;
        const bool more = un < nu;
        Unit tn = t;
        u32x4 rxn = {rx[0], rx[1], 0, rx[3]}, rwn = {rw[0], rw[1], 0, rw[3]};
        if (more) {
            tn = unit_of(a, un);
            rxn = descriptor(a.x + (size_t)tn.m0 * a.ldx_b, min(a.M - tn.m0, 256) * a.ldx_b);
            rwn = descriptor(a.w + (size_t)tn.n0 * a.ldw_b, min(a.N - tn.n0, 256) * a.ldw_b);
        }
        f32x4 acc[8][8];  // [W block][X block]
        {
            int ke = t.kt1 * 128, kd = min(t.kt0 * 128 + 256, ke), n = t.kt1 - t.kt0;
            const int k0n = tn.kt0 * 128, ken = tn.kt1 * 128;
            int xa, wa, tp = 0, t0 = 0;
#define K_LOOP_OPERANDS                                                                                               \
    : ACC_OUTPUTS,                                                                                                    \
      "+&{s[64:67]}"(rx), "+&{s[68:71]}"(rw), [xa] "=&v"(xa), [wa] "=&v"(wa), [sx] "+&s"(sx), [sw] "+&s"(sw),         \
      [sp] "+&s"(sp), [tp] "+&s"(tp), [t0] "+&s"(t0), [kd] "+&s"(kd), [ke] "+&s"(ke), [n] "+&s"(n)                    \
    : "{s[72:75]}"(rxn), "{s[76:79]}"(rwn), [k0n] "s"(k0n), [ken] "s"(ken), [ldsw] "s"(ldsw), [xlo0] "v"(xlo0),       \
      [xlo1] "v"(xlo1), [wlo0] "v"(wlo0), [wlo1] "v"(wlo1), [vx0] "v"(vx[0]), [vx1] "v"(vx[1]), [vx2] "v"(vx[2]),     \
      [vx3] "v"(vx[3]), [vx4] "v"(vx[4]), [vx5] "v"(vx[5]), [vx6] "v"(vx[6]), [vx7] "v"(vx[7]), [vw0] "v"(vw[0]),     \
      [vw1] "v"(vw[1]), [vw2] "v"(vw[2]), [vw3] "v"(vw[3]), [vw4] "v"(vw[4]), [vw5] "v"(vw[5]), [vw6] "v"(vw[6]),     \
      [vw7] "v"(vw[7])                                                                                                \
    : CLOBBERS
            if constexpr (GLU) asm volatile(K_LOOP(OFF_GLU) K_LOOP_OPERANDS);
            else asm volatile(K_LOOP(OFF_ROWS) K_LOOP_OPERANDS);
        }

        const Lane l = {t.m0, t.n0, wr, wc, lane & 15, lane >> 4};
        auto block = [&](int b, f32x4 (&v)[8]) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)  // named so that the others stay where they are: 256 do not fit beside the rest
                    asm("v_accvgpr_read_b32 %0, %1" : "=v"(v[j][r]) : "a"(acc[j][b][r]));
        };
        bool counted = false;  // exactly STORES vector memory operations behind the next unit's requests
        if (EPI == GEPI_F32 && a.slabs) {
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                f32x4 v[8];
                block(b, v);
                if (t.m0 + l.row(b) >= a.M) continue;
                float* out = a.part + ((size_t)t.slice * a.M + t.m0 + l.row(b)) * a.N;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = t.n0 + 128 * wc + 32 * q + 8 * l.g4;
                    if (n >= a.N) continue;
                    *reinterpret_cast<f32x4*>(out + n) = v[2 * q];
                    *reinterpret_cast<f32x4*>(out + n + 4) = v[2 * q + 1];
                }
            }
        } else if (t.slice >= 0) {
            // accumulator vector (b, j) of this lane at [8 b + j][thread]; 16-row blocks past M are skipped
            f32x4* out = reinterpret_cast<f32x4*>(a.part + ((size_t)(t.pos - a.whole) * a.splits + t.slice) * TILE_F) + tid;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                f32x4 v[8];
                block(b, v);
                if (t.m0 + 128 * wr + 16 * b >= a.M) continue;
#pragma unroll
                for (int j = 0; j < 8; ++j) out[(8 * b + j) * 256] = v[j];
            }
        } else if constexpr (WIDE) {
            counted = true;
            const int cols = GLU ? (a.N - t.n0) >> 1 : a.N - t.n0;  // of C from this tile's first
            const __amdgpu_buffer_rsrc_t rc =
                rsrc(reinterpret_cast<const bf16*>(a.c) + (size_t)t.m0 * a.ldc + (GLU ? t.n0 >> 1 : t.n0),
                     ((min(a.M - t.m0, 256) - 1) * a.ldc + min(cols, GLU ? 128 : 256)) * 2);
            int vo[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = (GLU ? 64 : 128) * wc + 32 * q + 8 * l.g4;
                vo[q] = c < cols ? l.row(0) * a.ldc * 2 + c * 2 : INT_MIN;  // past every range
            }
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                f32x4 v[8];
                block(b, v);
#pragma unroll
                for (int q = 0; q < (GLU ? 2 : 4); ++q) {
                    float o[8];
                    outputs<EPI>(v, q, a.glu, o);
                    const uint4 pk = pack8(o);
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{pk.x, pk.y, pk.z, pk.w}, rc, vo[q] + 32 * b * a.ldc, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                f32x4 v[8];
                block(b, v);
                store_rows<EPI>(a, l, b, v);
            }
        }
        if (!more) break;
        // X and W of the next unit's first K-tile have arrived: behind them are its second one and the stores
        if (counted) vm_wait<16 + STORES>();
        else vm_wait<0>();
        u = un;
        t = tn;
    }
    vm_wait<0>();  // nothing may arrive in LDS that another workgroup has by then
#ifdef MRSUM_CLOCK_STAMPS
    // in-kernel clock = shader ticks / 100 MHz ticks; lane 0's vector store to a buffer no other code reads
    __syncthreads();
    if (tid == 0) {
        const unsigned long long clk = __builtin_amdgcn_s_memtime() - clk0, rt = __builtin_amdgcn_s_memrealtime() - rt0;
        a.stamps[2 * blockIdx.x] = clk;
        a.stamps[2 * blockIdx.x + 1] = rt;
    }
#endif
}

// Adds the slices of the split tiles and runs the epilogue.  One workgroup per (tile, 2 x 16 rows): the eight vectors
// that every lane of gemm_bf16_kernel holds for one of its eight row blocks.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_bf16_tail_kernel(const GemmArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int t = blockIdx.x >> 3, b = blockIdx.x & 7;
    int tm, tn;
    tile_of(a.whole + t, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
    const Lane l = {tm * 256, tn * 256, w >> 1, w & 1, lane & 15, lane >> 4};
    if (l.m0 + 128 * l.wr + 16 * b >= a.M) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * TILE_F) + b * 8 * 256 + tid;
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = in[j * 256];
    for (int s = 1; s < a.splits; ++s) {
        in += TILE_F / 4;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] += in[j * 256];
    }
    store_rows<EPI>(a, l, b, v);
}

int gemm_bf16_grid(const GemmArgs& a) {
    const int nu = a.whole + (a.tiles_m * a.tiles_n - a.whole) * a.splits;
    // requests run up to two K-tiles into the next unit: with a single one a workgroup takes one unit only
    return a.kb / a.splits < 2 ? nu : std::min(nu, WGS);
}

void gemm_bf16_launch(const GemmArgs& a, int epi, hipStream_t s) {
    const dim3 grid(gemm_bf16_grid(a));
    const int rest = a.tiles_m * a.tiles_n - a.whole;
    const bool wide = a.ldc % 8 == 0 && (uintptr_t)a.c % 16 == 0 && (size_t)256 * a.ldc * 2 < (1u << 31);
#define GEMM_LAUNCH(E)                                                                \
    {                                                                                 \
        if (wide) gemm_bf16_kernel<E, true><<<grid, 256, 0, s>>>(a);                  \
        else gemm_bf16_kernel<E, false><<<grid, 256, 0, s>>>(a);                      \
        if (rest) gemm_bf16_tail_kernel<E><<<rest * 8, 256, 0, s>>>(a);               \
    }
    if (epi == GEPI_SWIGLU) GEMM_LAUNCH(GEPI_SWIGLU)
    else if (epi == GEPI_GELU) GEMM_LAUNCH(GEPI_GELU)
    else if (epi == GEPI_BF16) GEMM_LAUNCH(GEPI_BF16)
    else {
        gemm_bf16_kernel<GEPI_F32, false><<<grid, 256, 0, s>>>(a);
        if (rest && !a.slabs) gemm_bf16_tail_kernel<GEPI_F32><<<rest * 8, 256, 0, s>>>(a);
    }
#undef GEMM_LAUNCH
}
