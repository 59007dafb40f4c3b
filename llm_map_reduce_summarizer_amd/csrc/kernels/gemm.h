// What the two tile GEMMs share: gemm.hip (e4m3 operands, eight waves) and gemm_bf16.hip (bf16 operands, four waves).
#pragma once
#include "common.h"

enum { GEPI_BF16 = 0, GEPI_SWIGLU = 1, GEPI_GELU = 2, GEPI_F32 = 3 };

struct GemmArgs {
    const char* x;
    const char* w;
    void* c;
    const float* sx;  // fp8: per-row activation scale [M]
    const float* sw;  // fp8: per-row weight scale [N]
    int ldx_b, ldw_b, ldc;  // X / W row strides in bytes, C row stride in elements
    int M, N, kb;           // kb = K-tiles (128 bytes of every row each)
    int kbw;                // fp8, W's K-tiles: kb, or kb / 2 for two-term X (X tiles kt >= kbw re-read W tile kt - kbw)
    int rows;  // of a tile: 256, bf16 also 128, 160, 192, 224
    int tiles_m, tiles_n, group_m;
    int whole;    // raster positions below it run whole, the others in ``splits`` slices of K each
    int splits;
    float* part;  // [tiles - whole][splits][rows * 256] fp32 accumulators of the slices
    int slabs;    // GEPI_F32, every tile split: part is [splits][M][N] rows instead, for a consumer that adds the slabs
    GluArgs glu;  // GEPI_SWIGLU
#ifdef MRSUM_CLOCK_STAMPS
    unsigned long long* stamps;  // diagnostic build only (tools/gemm_clock.py): [grid][2] shader / 100 MHz ticks
#endif
};

// bf16 form (gemm_bf16.hip): epilogue ``epi`` of x . w^T; arguments as checked by mrsum_gemm
void gemm_bf16_launch(const GemmArgs& a, int epi, hipStream_t s);
// workgroups of that launch
int gemm_bf16_grid(const GemmArgs& a);

namespace {
constexpr int TILE_F = 256 * 256;  // accumulators of one tile

typedef __attribute__((address_space(3))) void* lds_ptr_t;

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, char* dst, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, voff, soff, 0, 0);
}

template <int N>
__device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// grouped raster of group_m tile rows
__device__ __forceinline__ void tile_of(int p, int tiles_m, int tiles_n, int group_m, int& tm, int& tn) {
    const int gsz = group_m * tiles_n;
    const int g = p / gsz, first = g * group_m;
    const int gm = min(tiles_m - first, group_m);
    const int within = p - g * gsz;
    tm = first + within % gm;
    tn = within / gm;
}
}  // namespace
