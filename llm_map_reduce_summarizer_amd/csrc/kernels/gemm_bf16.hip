// Large-M bf16 GEMM (prefill projections, LM head over many rows):
//
//     C[M, N] = X[M, K] . W[N, K]^T            X = activations, W = weights, both K-contiguous
//
// One output tile of 256 x 256 (or 128, 160, 192, 224 rows) at a time per workgroup of four waves, one wave per SIMD; wave
// (wr, wc) owns half the rows x 128 columns = up to 8 x 8 blocks of v_mfma_f32_16x16x32_bf16 in up to 256 accumulation
// registers.  What bounds it: LDS and the matrix cores.  A K-tile of 64 is 2048 cycles of MFMA per SIMD; eight waves of
// 128 x 64 read 192 KiB of fragments for it and fill 64 KiB by DMA, which is as many LDS cycles again, and took 2760 - 2850;
// four waves read 128 KiB and take 2200 - 2600.
// What else the fewer waves need is that nothing but the matrix cores is ever waited for, as no second wave covers a
// SIMD's waits, so the loop over K is written out:
//
//   * LDS: three images of W's K-tiles (256 rows x 128 B) and two of X's (three of 160 rows or fewer), each a ring.
//     Images arrive by LDS-DMA (buffer_load ... lds, 1 KiB = 8 rows per wave instruction) from a tile-local buffer
//     descriptor: rows past M / N are dropped by the descriptor's range check (their LDS rows hold stale bytes that
//     only feed masked outputs).  The bank swizzle is on the SOURCE address: 16-byte chunk c of row r sits at position
//     c ^ f(r), f taking all eight values over the rows that one fragment read touches.
//   * K-tile t: step 0 runs the MFMAs of k 0 - 31 while the fragments of k 32 - 63 come from LDS into the other
//     register set; then the one wait and barrier of the K-tile: every wave has its fragments of t, and X, W(t + 1) have
//     arrived; step 1 runs k 32 - 63 while the first fragments of t + 1 are read, and asks for the X that goes where X(t)
//     was and the first half of W(t + 3), which goes where W(t) was; its second half is asked for in step 0 of t + 1.  W,
//     which comes from further away where rows are few, has one and a half K-tiles to arrive, X one (of few rows two).
//     Requests two K-tiles ahead in a common ring of five images left the last of W half a K-tile: 305 x 28672 x 4096
//     91 us, 80 in tiles of 160 rows; so 87 and 72, and W past the caches (nt, where no other round reads it) 70.
//   * the workgroups stay for all their tiles, and the requests run on into the next tile (or slice of K), whose first
//     K-tiles arrive while the epilogue runs.  The epilogue keeps out of LDS for that: W's rows are dealt to the MFMA
//     rows so that a lane ends with 8 consecutive output columns (gate and up of the same columns for GLU) of a row, one
//     16-byte store, 64 bytes in a row by four lanes.
//   * the MFMA computes the transposed tile (A = W fragment, B = X fragment); column blocks go back and forth over the row
//     blocks, so that a neighbour's operand stays.
//   * split tail: tiles behind the last whole round of 256 (all of them where M and N are small) would leave most CUs
//     idle for a full K loop, so each is cut into S slices of K.  A slice writes its fp32 accumulators to scratch in
//     register order (lane-contiguous 16-B stores) and gemm_bf16_tail_kernel adds them in slice order and runs the
//     epilogue: a second launch and no ticket, so results do not depend on arrival and concurrent streams share
//     nothing.  Rows of a tile and slices: mrsum_gemm_plan.
//
// Measured, eight waves (two 64 KiB tiles of LDS, two barriers a quarter of a K-tile) -> this, us: 18234 x 28672 x 4096 with
// GLU 3439 -> 3015 (1420 TFLOP/s), 18234 x 4096 x 14336 1546 -> 1421 (1507), 18234 x 6144 x 4096 685 -> 640, 1967 x 18432 x
// 4096 with gelu 258 -> 238.  The large ones run at the clock that the card's power allows (1.8 - 1.9 of 2.4 GHz): requests
// earlier or later, or reads closer together, change them by less than 1 %.
#include "gemm.h"

namespace {
constexpr int IMAGE = 256 * 128, X0 = 3 * IMAGE;  // a K-tile of W; X's images behind W's three
constexpr int x_image(int nb) { return nb * 4096; }
constexpr int x_slots(int nb) { return nb <= 5 ? 3 : 2; }
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
// one row block against all column blocks, with room for reads and a request after every two
#define ROW(M, s, b, a0, a1, a2, a3)  M(s, 0, b) M(s, 1, b) a0 M(s, 2, b) M(s, 3, b) a1 M(s, 4, b) M(s, 5, b) a2 M(s, 6, b) M(s, 7, b) a3
#define BACK(M, s, b, a0, a1, a2, a3) M(s, 7, b) M(s, 6, b) a0 M(s, 5, b) M(s, 4, b) a1 M(s, 3, b) M(s, 2, b) a2 M(s, 1, b) M(s, 0, b) a3
#define RX(s, b) "ds_read_b128 " XF(s, b) ", %[xa] offset:" STR(2048 * b) "\n"
#define RW(s, j, off) "ds_read_b128 " WF(s, j) ", %[wa] offset:" STR(128 * off(j)) "\n"
// requests; m0 moves on behind each, behind X's last to W's first place
#define REQ(v, r, k, nt, m) "buffer_load_dwordx4 %[" v "], " r ", %[" k "] offen" nt " lds\ns_add_u32 m0, " m "\n"
#define DX(p) REQ("vx" #p, "s[64:67]", "kx", "", "m0, 0x400")
#define DXL(p) REQ("vx" #p, "s[64:67]", "kx", "", "%[tw], %[ldsw]")
#define DW(p) REQ("vw" #p, "s[68:71]", "kw", "", "m0, 0x400")
#define DWN(p) REQ("vw" #p, "s[68:71]", "kw", " nt", "m0, 0x400")
#define READ_AT(x, w) "v_add_u32 %[xa], %[sx], %[" x "]\nv_add_u32 %[wa], %[sw], %[" w "]\n"
#define NEXT(r, size, end) "s_add_u32 %[" r "], %[" r "], " size "\ns_cmp_ge_u32 %[" r "], " end "\ns_cselect_b32 %[" r "], 0, %[" r "]\n"
// half a K-tile: the MFMAs of fragment set s row block by row block, in between the reads of set o as early as LDS serves
// them (one for two MFMAs), the last row block covering the last ones, and the requests q0 ..
#define STEP_8(M, s, o, off, q0, q1, q2, q3, q4, q5, q6, q7, q8, q9, q10, q11)              \
    ROW(M, s, 0, RX(o, 0), RX(o, 1) q0, RX(o, 2), q1)                                       \
    BACK(M, s, 1, RX(o, 3), RX(o, 4) q2, RX(o, 5), q3)                                      \
    ROW(M, s, 2, RX(o, 6), RX(o, 7) q4, RW(o, 0, off), q5)                                  \
    BACK(M, s, 3, RW(o, 1, off), RW(o, 2, off) q6, RW(o, 3, off), q7)                       \
    ROW(M, s, 4, RW(o, 4, off), RW(o, 5, off), , q8)                                        \
    BACK(M, s, 5, RW(o, 6, off), RW(o, 7, off), , q9)                                       \
    ROW(M, s, 6, , , , q10)                                                                 \
    BACK(M, s, 7, , , , q11)
#define STEP_7(M, s, o, off, q0, q1, q2, q3, q4, q5, q6, q7, q8, q9, q10, q11)              \
    ROW(M, s, 0, RX(o, 0), RX(o, 1) q0, RX(o, 2), q1)                                       \
    BACK(M, s, 1, RX(o, 3), RX(o, 4) q2, RX(o, 5), q3)                                      \
    ROW(M, s, 2, RX(o, 6), RW(o, 0, off) q4, RW(o, 1, off), q5)                             \
    BACK(M, s, 3, RW(o, 2, off), RW(o, 3, off) q6, RW(o, 4, off), q7)                       \
    ROW(M, s, 4, RW(o, 5, off), RW(o, 6, off), RW(o, 7, off), q8)                           \
    BACK(M, s, 5, , q9, , q10)                                                              \
    ROW(M, s, 6, , q11, , )
#define STEP_6(M, s, o, off, q0, q1, q2, q3, q4, q5, q6, q7, q8, q9, q10, q11)              \
    ROW(M, s, 0, RX(o, 0), RX(o, 1) q0, RX(o, 2), q1)                                       \
    BACK(M, s, 1, RX(o, 3), RX(o, 4) q2, RX(o, 5), q3)                                      \
    ROW(M, s, 2, RW(o, 0, off), RW(o, 1, off) q4, RW(o, 2, off), q5)                        \
    BACK(M, s, 3, RW(o, 3, off), RW(o, 4, off) q6, RW(o, 5, off), q7)                       \
    ROW(M, s, 4, RW(o, 6, off), RW(o, 7, off) q8, , q9)                                     \
    BACK(M, s, 5, , q10, , q11)
#define STEP_5(M, s, o, off, q0, q1, q2, q3, q4, q5, q6, q7, q8, q9, q10, q11)              \
    ROW(M, s, 0, RX(o, 0), RX(o, 1) q0, RX(o, 2), q1)                                       \
    BACK(M, s, 1, RX(o, 3), RX(o, 4) q2, RW(o, 0, off), q3)                                 \
    ROW(M, s, 2, RW(o, 1, off), RW(o, 2, off) q4, RW(o, 3, off), q5)                        \
    BACK(M, s, 3, RW(o, 4, off), RW(o, 5, off) q6, RW(o, 6, off), RW(o, 7, off) q7)         \
    ROW(M, s, 4, q8, q9, q10, q11)
#define STEP_4(M, s, o, off, q0, q1, q2, q3, q4, q5, q6, q7, q8, q9, q10, q11)              \
    ROW(M, s, 0, RX(o, 0), RX(o, 1) q0, RX(o, 2), RX(o, 3) q1)                              \
    BACK(M, s, 1, RW(o, 0, off), RW(o, 1, off) q2, RW(o, 2, off), RW(o, 3, off) q3)         \
    ROW(M, s, 2, RW(o, 4, off), RW(o, 5, off) q4, RW(o, 6, off), RW(o, 7, off) q5)          \
    BACK(M, s, 3, q6, q7, q8, q9 q10 q11)
// step 1 asks for X and the first half of W, step 0 of the next K-tile for W's second half
#define ASK1_8 DX(0), DX(1), DX(2), DX(3), DX(4), DX(5), DX(6), DXL(7), DW(0), DW(1), DW(2), DW(3)
#define ASK1_7 DX(0), DX(1), DX(2), DX(3), DX(4), DX(5), DXL(6), DW(0), DW(1), DW(2), DW(3),
#define ASK1_6 DX(0), DX(1), DX(2), DX(3), DX(4), DXL(5), DW(0), DW(1), DW(2), DW(3), ,
#define ASK1_5 DX(0), DX(1), DX(2), DX(3), DXL(4), DW(0), DW(1), DW(2), DW(3), , ,
#define ASK1_4 DX(0), DX(1), DX(2), DXL(3), DW(0), DW(1), DW(2), DW(3), , , ,
#define ASK0_8 , DW(4), , DW(5), , DW(6), , DW(7), , , ,
#define ASK0_7 ASK0_8
#define ASK0_6 ASK0_8
#define ASK0_5 ASK0_8
#define ASK0_4 ASK0_8
// with W past the caches
#define ASK1_6N DX(0), DX(1), DX(2), DX(3), DX(4), DXL(5), DWN(0), DWN(1), DWN(2), DWN(3), ,
#define ASK1_5N DX(0), DX(1), DX(2), DX(3), DXL(4), DWN(0), DWN(1), DWN(2), DWN(3), , ,
#define ASK1_4N DX(0), DX(1), DX(2), DXL(3), DWN(0), DWN(1), DWN(2), DWN(3), , , ,
#define ASK0_6N , DWN(4), , DWN(5), , DWN(6), , DWN(7), , , ,
#define ASK0_5N ASK0_6N
#define ASK0_4N ASK0_6N
#define EXPAND(...) __VA_ARGS__
#define STEP0(NB, ASK, M, off) READ_AT("xlo1", "wlo1") "s_add_u32 m0, %[tw], %[ldsw4]\n" EXPAND(STEP_##NB EXPAND((M, 0, 1, off, ASK0_##ASK)))
#define STEP1(NB, ASK, off) READ_AT("xlo0", "wlo0") "s_add_u32 m0, %[tx], %[ldsx]\n" EXPAND(STEP_##NB EXPAND((MF, 1, 0, off, ASK1_##ASK)))
#define READ_X_4 RX(0, 0) RX(0, 1) RX(0, 2) RX(0, 3)
#define READ_X_5 READ_X_4 RX(0, 4)
#define READ_X_6 READ_X_5 RX(0, 5)
#define READ_X_7 READ_X_6 RX(0, 6)
#define READ_X_8 READ_X_7 RX(0, 7)
// the requests of an operand have passed this unit's last K-tile: on to the next unit's first
#define FOLLOW(k, ke, r0, r1, n0, n1, label)                                                \
    "s_cmp_lg_u32 %[" k "], %[" ke "]\ns_cbranch_scc1 " label "f\n"                         \
    "s_mov_b64 " r0 ", " n0 "\ns_mov_b64 " r1 ", " n1 "\n"                                  \
    "s_mov_b32 %[" k "], %[k0n]\ns_mov_b32 %[" ke "], %[ken]\n" label ":\n"
#define K_LOOP(NB, ASK, off)                                                                \
    "s_barrier\n" READ_AT("xlo0", "wlo0") READ_X_##NB                                       \
    RW(0, 0, off) RW(0, 1, off) RW(0, 2, off) RW(0, 3, off)                                 \
    RW(0, 4, off) RW(0, 5, off) RW(0, 6, off) RW(0, 7, off)                                 \
    "s_waitcnt lgkmcnt(0)\n" STEP0(NB, ASK, MZ, off)                                        \
    "s_waitcnt vmcnt(%[w0]) lgkmcnt(0)\ns_branch 2f\n"                                      \
    "1:\ns_waitcnt lgkmcnt(0)\n" STEP0(NB, ASK, MF, off)                                    \
    "s_waitcnt vmcnt(%[w1]) lgkmcnt(0)\n2:\ns_barrier\n"                                    \
    "s_mov_b32 %[tx], %[sx]\ns_mov_b32 %[tw], %[sw]\n"                                      \
    NEXT("sx", "%[xi]", "%[xe]") NEXT("sw", "0x8000", "0x18000")                            \
    "s_add_u32 %[kw], %[kw], 0x80\n"                                                        \
    FOLLOW("kx", "kex", "s[64:65]", "s[66:67]", "s[72:73]", "s[74:75]", "3")                \
    FOLLOW("kw", "kew", "s[68:69]", "s[70:71]", "s[76:77]", "s[78:79]", "4")                \
    STEP1(NB, ASK, off)                                                                     \
    "s_add_u32 %[kx], %[kx], 0x80\ns_sub_u32 %[n], %[n], 1\ns_cmp_lg_u32 %[n], 0\n"         \
    "s_cbranch_scc1 1b\ns_waitcnt lgkmcnt(0)\ns_nop 15\n"
// the W row of MFMA row a = lane & 15 of block j is OFF(j) + (8 or 16) (a >> 2) + (a & 3)
#define OFF_ROWS(j) (32 * (j >> 1) + 4 * (j & 1))
#define OFF_GLU(j) (64 * (j >> 2) + 4 * (j & 3))
#define ACC_B0 \
    "={a[0:3]}"(acc[0][0]), "={a[32:35]}"(acc[1][0]), "={a[64:67]}"(acc[2][0]), "={a[96:99]}"(acc[3][0]), \
    "={a[128:131]}"(acc[4][0]), "={a[160:163]}"(acc[5][0]), "={a[192:195]}"(acc[6][0]), "={a[224:227]}"(acc[7][0])
#define ACC_B1 \
    "={a[4:7]}"(acc[0][1]), "={a[36:39]}"(acc[1][1]), "={a[68:71]}"(acc[2][1]), "={a[100:103]}"(acc[3][1]), \
    "={a[132:135]}"(acc[4][1]), "={a[164:167]}"(acc[5][1]), "={a[196:199]}"(acc[6][1]), "={a[228:231]}"(acc[7][1])
#define ACC_B2 \
    "={a[8:11]}"(acc[0][2]), "={a[40:43]}"(acc[1][2]), "={a[72:75]}"(acc[2][2]), "={a[104:107]}"(acc[3][2]), \
    "={a[136:139]}"(acc[4][2]), "={a[168:171]}"(acc[5][2]), "={a[200:203]}"(acc[6][2]), "={a[232:235]}"(acc[7][2])
#define ACC_B3 \
    "={a[12:15]}"(acc[0][3]), "={a[44:47]}"(acc[1][3]), "={a[76:79]}"(acc[2][3]), "={a[108:111]}"(acc[3][3]), \
    "={a[140:143]}"(acc[4][3]), "={a[172:175]}"(acc[5][3]), "={a[204:207]}"(acc[6][3]), "={a[236:239]}"(acc[7][3])
#define ACC_B4 \
    "={a[16:19]}"(acc[0][4]), "={a[48:51]}"(acc[1][4]), "={a[80:83]}"(acc[2][4]), "={a[112:115]}"(acc[3][4]), \
    "={a[144:147]}"(acc[4][4]), "={a[176:179]}"(acc[5][4]), "={a[208:211]}"(acc[6][4]), "={a[240:243]}"(acc[7][4])
#define ACC_B5 \
    "={a[20:23]}"(acc[0][5]), "={a[52:55]}"(acc[1][5]), "={a[84:87]}"(acc[2][5]), "={a[116:119]}"(acc[3][5]), \
    "={a[148:151]}"(acc[4][5]), "={a[180:183]}"(acc[5][5]), "={a[212:215]}"(acc[6][5]), "={a[244:247]}"(acc[7][5])
#define ACC_B6 \
    "={a[24:27]}"(acc[0][6]), "={a[56:59]}"(acc[1][6]), "={a[88:91]}"(acc[2][6]), "={a[120:123]}"(acc[3][6]), \
    "={a[152:155]}"(acc[4][6]), "={a[184:187]}"(acc[5][6]), "={a[216:219]}"(acc[6][6]), "={a[248:251]}"(acc[7][6])
#define ACC_B7 \
    "={a[28:31]}"(acc[0][7]), "={a[60:63]}"(acc[1][7]), "={a[92:95]}"(acc[2][7]), "={a[124:127]}"(acc[3][7]), \
    "={a[156:159]}"(acc[4][7]), "={a[188:191]}"(acc[5][7]), "={a[220:223]}"(acc[6][7]), "={a[252:255]}"(acc[7][7])
#define ACC_4 ACC_B0, ACC_B1, ACC_B2, ACC_B3
#define ACC_5 ACC_4, ACC_B4
#define ACC_6 ACC_5, ACC_B5
#define ACC_7 ACC_6, ACC_B6
#define ACC_8 ACC_7, ACC_B7
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
template <int NB>
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
    t.m0 = tm * 32 * NB;
    t.n0 = tn * 256;
    return t;
}

// Where a lane's outputs go: row block b is rows m0 + 16 b + (lane & 15); column group q (4, GLU 2) is 8 columns from col(q).
template <int NB>
struct Lane {
    int m0, n0, wr, wc, r16, g4;
    __device__ __forceinline__ int row(int b) const { return 16 * NB * wr + 16 * b + r16; }  // within the tile
};

// The outputs of column group q from a row block's accumulators v[j] (W block j).
// GLU divides: the hardware reciprocal is 1 - 2 % of the kernel faster (18234 x 28672 x 4096 2954 -> 2900 us, 305 rows 69.8 ->
// 69.0) but a bit less exact, and scaled to reach every exponential it loses the bits of gates under 2^-94.
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
template <int EPI, int NB>
__device__ __forceinline__ void store_rows(const GemmArgs& a, const Lane<NB>& l, int b, const f32x4 (&v)[8]) {
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
// descriptor in a fixed number of 16-byte stores, which the next tile's first wait can count past.  NT: W past the caches.
template <int EPI, bool WIDE, int NB, bool NT>
__global__ __launch_bounds__(256, 1) void gemm_bf16_kernel(const GemmArgs a) {
    static_assert(!(WIDE && EPI == GEPI_F32), "fp32 rows leave by store_rows");
#ifdef MRSUM_CLOCK_STAMPS
    const unsigned long long clk0 = __builtin_amdgcn_s_memtime(), rt0 = __builtin_amdgcn_s_memrealtime();
#endif
    constexpr bool GLU = EPI == GEPI_SWIGLU;
    constexpr int ROWS = 32 * NB, STORES = NB * (GLU ? 2 : 4);
    constexpr int XI = x_image(NB), XS = x_slots(NB);
    // requests behind X and W of the K-tile t + 1 in the middle of t, and in the first K-tile of a later unit, where the
    // stores of the unit before stand in between
    constexpr int AHEAD = 8 + (XS == 3 ? NB : 0), AHEAD0 = AHEAD + (WIDE ? STORES : 0);
    __shared__ __attribute__((aligned(1024))) char lds[X0 + XS * XI];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w >> 1, wc = w & 1;
    const int nu = units(a);

    // staging: wave w fills a quarter of an image's rows in pieces of 8; position lane & 7 of row r takes chunk
    // (lane & 7) ^ f(r), f over bits 1 - 3 of an X row and the bits of a W row that a fragment read spans
    int vx[NB], vw[8];
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        const int r = 8 * (NB * w + p) + (lane >> 3);
        vx[p] = r * a.ldx_b + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int r = 64 * w + 8 * p + (lane >> 3);
        const int fw = ((r >> 1) & 1) | (((r >> (GLU ? 4 : 3)) & 3) << 1);
        vw[p] = r * a.ldw_b + (((lane & 7) ^ fw) << 4);
    }
    // fragment reads: row lane & 15 of a block, chunk lane >> 4 (step 0) or 4 + (lane >> 4) (step 1)
    const int fr = lane & 15, pos0 = ((lane >> 4) ^ (fr >> 1)) << 4;
    const int base = (int)(uintptr_t)(lds_ptr_t)lds;
    const int xlo0 = base + X0 + (16 * NB * wr + fr) * 128 + pos0;
    const int wlo0 = base + (128 * wc + (GLU ? 16 : 8) * (fr >> 2) + (fr & 3)) * 128 + pos0;
    const int xlo1 = xlo0 ^ 64, wlo1 = wlo0 ^ 64, ldsw = base + w * 8192, ldsw4 = ldsw + 4096, ldsx = base + X0 + w * NB * 1024;

    Unit t = unit_of<NB>(a, blockIdx.x);
    u32x4 rx = descriptor(a.x + (size_t)t.m0 * a.ldx_b, min(a.M - t.m0, ROWS) * a.ldx_b);
    u32x4 rw = descriptor(a.w + (size_t)t.n0 * a.ldw_b, min(a.N - t.n0, 256) * a.ldw_b);
    {  // the first unit's first K-tiles, in the loop's order; past a short one its last again, which nothing reads
        const __amdgpu_buffer_rsrc_t bx = rsrc(a.x + (size_t)t.m0 * a.ldx_b, min(a.M - t.m0, ROWS) * a.ldx_b);
        const __amdgpu_buffer_rsrc_t bw = rsrc(a.w + (size_t)t.n0 * a.ldw_b, min(a.N - t.n0, 256) * a.ldw_b);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int k = min(t.kt0 + i, t.kt1 - 1) * 128;
            if (i < XS)
#pragma unroll
                for (int p = 0; p < NB; ++p) dma16(bx, lds + X0 + i * XI + (w * NB + p) * 1024, vx[p], k);
#pragma unroll
            for (int p = 0; p < (i < 2 ? 8 : 4); ++p) dma16(bw, lds + i * IMAGE + w * 8192 + p * 1024, vw[p], k);
        }
    }
    vm_wait<AHEAD - 4>();  // all but what the middle of a K-tile does not wait for
    int sx = 0, sw = 0, tw = 2 * IMAGE;  // images of X(t) and W(t), and of the W that is asked for

    for (int u = blockIdx.x;;) {
        // what follows: the next unit, or a descriptor that drops every request
        const int un = u + gridDim.x;
        const bool more = un < nu;
        Unit tn = t;
        u32x4 rxn = {rx[0], rx[1], 0, rx[3]}, rwn = {rw[0], rw[1], 0, rw[3]};
        if (more) {
            tn = unit_of<NB>(a, un);
            rxn = descriptor(a.x + (size_t)tn.m0 * a.ldx_b, min(a.M - tn.m0, ROWS) * a.ldx_b);
            rwn = descriptor(a.w + (size_t)tn.n0 * a.ldw_b, min(a.N - tn.n0, 256) * a.ldw_b);
        }
        f32x4 acc[8][NB];  // [W block][X block]
        {
            int kex = t.kt1 * 128, kew = kex, n = t.kt1 - t.kt0;
            int kx = min(t.kt0 * 128 + XS * 128, kex), kw = min(t.kt0 * 128 + 256, kew - 128);
            const int k0n = tn.kt0 * 128, ken = tn.kt1 * 128;
            int xa, wa, tx = 0;
#define X_4 [vx0] "v"(vx[0]), [vx1] "v"(vx[1]), [vx2] "v"(vx[2]), [vx3] "v"(vx[3])
#define X_5 X_4, [vx4] "v"(vx[4])
#define X_6 X_5, [vx5] "v"(vx[5])
#define X_7 X_6, [vx6] "v"(vx[6])
#define X_8 X_7, [vx7] "v"(vx[7])
#define K_LOOP_OPERANDS(NB)                                                                                           \
    : ACC_##NB, "+&{s[64:67]}"(rx), "+&{s[68:71]}"(rw), [xa] "=&v"(xa), [wa] "=&v"(wa), [sx] "+&s"(sx),               \
      [sw] "+&s"(sw), [tx] "+&s"(tx), [tw] "+&s"(tw), [kx] "+&s"(kx), [kex] "+&s"(kex), [kw] "+&s"(kw),               \
      [kew] "+&s"(kew), [n] "+&s"(n)                                                                                  \
    : "{s[72:75]}"(rxn), "{s[76:79]}"(rwn), [k0n] "s"(k0n), [ken] "s"(ken), [ldsx] "s"(ldsx), [ldsw] "s"(ldsw),       \
      [ldsw4] "s"(ldsw4), [xi] "n"(XI), [xe] "n"(XS * XI), [w0] "n"(AHEAD0), [w1] "n"(AHEAD),                         \
      [xlo0] "v"(xlo0), [xlo1] "v"(xlo1), [wlo0] "v"(wlo0), [wlo1] "v"(wlo1), X_##NB, [vw0] "v"(vw[0]),               \
      [vw1] "v"(vw[1]), [vw2] "v"(vw[2]), [vw3] "v"(vw[3]), [vw4] "v"(vw[4]), [vw5] "v"(vw[5]), [vw6] "v"(vw[6]),     \
      [vw7] "v"(vw[7])                                                                                                \
    : CLOBBERS
#define RUN_K(NB_, ASK, NT_)                                                              \
    if constexpr (NB == NB_ && NT == NT_) {                                               \
        if constexpr (GLU) asm volatile(K_LOOP(NB_, ASK, OFF_GLU) K_LOOP_OPERANDS(NB_));  \
        else asm volatile(K_LOOP(NB_, ASK, OFF_ROWS) K_LOOP_OPERANDS(NB_));               \
    }
            RUN_K(4, 4N, true) RUN_K(5, 5N, true) RUN_K(6, 6N, true)
            RUN_K(4, 4, false) RUN_K(5, 5, false) RUN_K(6, 6, false) RUN_K(7, 7, false) RUN_K(8, 8, false)
        }

        const Lane<NB> l = {t.m0, t.n0, wr, wc, lane & 15, lane >> 4};
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
            for (int b = 0; b < NB; ++b) {
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
            f32x4* out = reinterpret_cast<f32x4*>(a.part + ((size_t)(t.pos - a.whole) * a.splits + t.slice) * (ROWS * 256)) + tid;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 v[8];
                block(b, v);
                if (t.m0 + 16 * NB * wr + 16 * b >= a.M) continue;
#pragma unroll
                for (int j = 0; j < 8; ++j) out[(8 * b + j) * 256] = v[j];
            }
        } else if constexpr (WIDE) {
            counted = true;
            const int cols = GLU ? (a.N - t.n0) >> 1 : a.N - t.n0;  // of C from this tile's first
            const __amdgpu_buffer_rsrc_t rc =
                rsrc(reinterpret_cast<const bf16*>(a.c) + (size_t)t.m0 * a.ldc + (GLU ? t.n0 >> 1 : t.n0),
                     ((min(a.M - t.m0, ROWS) - 1) * a.ldc + min(cols, GLU ? 128 : 256)) * 2);
            int vo[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = (GLU ? 64 : 128) * wc + 32 * q + 8 * l.g4;
                vo[q] = c < cols ? l.row(0) * a.ldc * 2 + c * 2 : INT_MIN;  // past every range
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
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
            for (int b = 0; b < NB; ++b) {
                f32x4 v[8];
                block(b, v);
                store_rows<EPI, NB>(a, l, b, v);
            }
        }
        if (!more) break;
        // the next unit's first K-tile has arrived in the middle of this one's last; its second one is waited for past the
        // stores, where their number is known
        if (!counted) vm_wait<0>();
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
template <int EPI, int NB>
__global__ __launch_bounds__(256) void gemm_bf16_tail_kernel(const GemmArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int t = blockIdx.x / NB, b = blockIdx.x % NB;
    int tm, tn;
    tile_of(a.whole + t, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
    const Lane<NB> l = {tm * 32 * NB, tn * 256, w >> 1, w & 1, lane & 15, lane >> 4};
    if (l.m0 + 16 * NB * l.wr + 16 * b >= a.M) return;
    const f32x4* in = reinterpret_cast<const f32x4*>(a.part + (size_t)t * a.splits * (32 * NB * 256)) + b * 8 * 256 + tid;
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = in[j * 256];
    for (int s = 1; s < a.splits; s += 3) {  // three slices in flight: one at a time paid memory's latency for each
        f32x4 p[3][8];
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j) p[k][j] = in[(size_t)min(s + k, a.splits - 1) * (32 * NB * 64) + j * 256];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (s + k < a.splits)
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] += p[k][j];
    }
    store_rows<EPI, NB>(a, l, b, v);
}

int gemm_bf16_grid(const GemmArgs& a) {
    const int nu = a.whole + (a.tiles_m * a.tiles_n - a.whole) * a.splits;
    // requests run up to three K-tiles into the next unit: of shorter units a workgroup takes one only
    return a.kb / a.splits < 3 ? nu : std::min(nu, WGS);
}

template <int NB, bool NT>
static void launch_form(const GemmArgs& a, int epi, hipStream_t s) {
    const dim3 grid(gemm_bf16_grid(a));
    const int rest = a.tiles_m * a.tiles_n - a.whole;
    const bool wide = a.ldc % 8 == 0 && (uintptr_t)a.c % 16 == 0 && (size_t)256 * a.ldc * 2 < (1u << 31);
#define GEMM_LAUNCH(E)                                                                \
    {                                                                                 \
        if (wide) gemm_bf16_kernel<E, true, NB, NT><<<grid, 256, 0, s>>>(a);          \
        else gemm_bf16_kernel<E, false, NB, NT><<<grid, 256, 0, s>>>(a);              \
        if (rest) gemm_bf16_tail_kernel<E, NB><<<rest * NB, 256, 0, s>>>(a);          \
    }
    if (epi == GEPI_SWIGLU) GEMM_LAUNCH(GEPI_SWIGLU)
    else if (epi == GEPI_GELU) GEMM_LAUNCH(GEPI_GELU)
    else if (epi == GEPI_BF16) GEMM_LAUNCH(GEPI_BF16)
    else {
        gemm_bf16_kernel<GEPI_F32, false, NB, NT><<<grid, 256, 0, s>>>(a);
        if (rest && !a.slabs) gemm_bf16_tail_kernel<GEPI_F32, NB><<<rest * NB, 256, 0, s>>>(a);
    }
#undef GEMM_LAUNCH
}

// W of up to 192 rows goes past the caches where all row tiles of a column are neighbours in the raster, so that no later
// round reads it again.  us, through the caches -> past them: 305 x 24576 x 4096 (2 row tiles) 67.6 -> 64.2, 600 x 8192 x 4096
// (4) 47.4 -> 46.5; but 903 x 24576 x 4096 (5) 149 -> 156, 903 x 8192 x 4096 (8) 57 -> 63, 1300 x 6144 x 4096 (9) 61 -> 68, 4096 x
// 2176 x 4096 (26) 61 -> 70.
template <int NB>
static void launch_rows(const GemmArgs& a, int epi, hipStream_t s) {
    if constexpr (NB <= 6)
        if (a.tiles_m <= a.group_m) return launch_form<NB, true>(a, epi, s);
    launch_form<NB, false>(a, epi, s);
}

void gemm_bf16_launch(const GemmArgs& a, int epi, hipStream_t s) {
    switch (a.rows) {
        case 128: launch_rows<4>(a, epi, s); break;
        case 160: launch_rows<5>(a, epi, s); break;
        case 192: launch_rows<6>(a, epi, s); break;
        case 224: launch_rows<7>(a, epi, s); break;
        default: launch_rows<8>(a, epi, s); break;
    }
}

// Rows of a tile, raster position from which tiles run in slices of K, and the slices (1: none do) of an M x N product of kb
// K-tiles: the cheapest by a model of the kernel, fitted to 21 shapes (N 1024 - 28672, K 512 - 22528) at 47 row counts from 3 to
// 7615.  There and at 6 other shapes it loses 1 % on average against the best height and slices, 20 % at most (200 x 28672 x 4096
// with GLU: 72 us in 224 rows and two slices, 60 in 128 whole).  256 rows at their best slices are 17 % slower on average at M 130 -
// 1000, 11 % up to 4000 and 4 % beyond: M 305, N 28672, K 4096 91 us (160 rows: 67), M 1967, N 4096, K 4096 68 (128: 56).
MRSUM_API int mrsum_gemm_plan(int M, int N, int kb, int* out) {
    // us a K-tile: few workgroups at work, and all CUs (the clock that power allows, and what all ask of memory)
    struct Height { int rows; float few, full; };
    static constexpr Height H[5] = {{256, .962f, 1.294f}, {224, .928f, 1.157f}, {192, .867f, 1.059f}, {160, .783f, .958f}, {128, .472f, .884f}};
    const int tn = ceil_div(N, 256);
    float best = INFINITY;
    for (const Height& h : H) {
        const int tm = ceil_div(M, h.rows), tiles = tm * tn, rest = tiles % WGS;
        const float epilogue = 3.13f * h.rows / 256;
        // slices below 32 K-tiles: a whole loop is as short as the second launch, and a row's sum the same whichever rows
        // run with it.  They fill one round, or two with up to three a tile.
        const int most = kb < 32 || !rest ? 1 : std::min(std::max(WGS / rest, std::min(3, 2 * WGS / rest)), kb / 4);
        for (int s = 1; s <= std::max(1, most); ++s) {
            const float ks = (float)kb / s;
            const int n = rest * s, last = n % WGS;
            float t = (tiles / WGS) * (kb * h.full + epilogue) + (n / WGS) * (ks * h.full + epilogue);
            const float load = last ? last / (float)WGS : 1.f;
            if (last) t += ks * (h.few + (h.full - h.few) * load) + epilogue;
            // a round of stores on the last CUs: 903 x 8192 x 512 17.6 us, 13.0 in 192 tiles
            if (s == 1) t += 7.1f * std::max(0.f, load - .764f);
            if (s > 1) {  // the second launch, and accumulators written and read again: dearer beyond what the L2s hold
                const float mb = (float)n * (16 * ceil_div(M, 16)) / tm * 1024e-6f;
                t += 3.4f + .44f * s + .12f * mb + .178f * std::max(0.f, mb - 28.7f);
            }
            if (t < best) {
                best = t;
                out[0] = h.rows;
                out[1] = s > 1 ? tiles - rest : tiles;
                out[2] = s;
            }
        }
    }
    return 0;
}
