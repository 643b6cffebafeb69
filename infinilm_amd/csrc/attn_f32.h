// What the kernels of the 32-bit path's attention share (attn_f32.hip, attn_f32_tile.hip): the chunks that fix the order of every
// sum, and the fold of their partial results.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define FA_CHUNK 128
#define FA_TILES (FA_CHUNK / 16)
#define FT_TOKENS 8   // most tokens a tile (attn_f32_tile.hip)
#define FA_WS_PAD 4   // a partial result is d outputs, its maximum, its sum and two unused floats (16-byte rows)

__device__ __forceinline__ f32x4 fa_mfma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// (M, L, ACC) <- fold of (M, L, ACC) and a chunk's (m, l, acc): explicit multiply-adds, the same in all
// launch shapes and in the fold kernel
__device__ __forceinline__ void fa_fold_scales(float& M, float& L, float m, float l, float& a, float& b) {
    const float Mn = fmaxf(M, m);
    a = expf(M - Mn);
    b = expf(m - Mn);
    L = fmaf(L, a, l * b);
    M = Mn;
}

// Folds partial results (attn_f32.hip): ws[((row * nh + h) * nchunks + chunk) * (d + FA_WS_PAD)], rows: eight of each of the n_tiles tiles (first token, count:
// up to count of them hold something), then n_rows single tokens
int fa_fold(float* out, const float* ws, const int* pos, const int* tiles, int n_tiles, const int* rows, int first, int n_rows, int nh, int d, int nchunks,
            int out_stride, int reach, hipStream_t stream);
extern "C" int ilm_attn_f32_tile_ok(int d, int page);   // attn_f32_tile.hip
