// Float products on the bfloat16 matrix cores.  A float has 24 bits of mantissa, a bfloat16 eight: x = h + m + l in
// bfloat16 is exact (h cut off, so that no float overflows; m and l rounded to nearest), a product of two pieces is
// exact in the instruction's float sum, and of the nine products the three smallest (m l, l m, l l: below 2^-24
// of the whole, of either sign) are left out.  Six v_mfma_f32_16x16x32_bf16 do the work of eight
// v_mfma_f32_16x16x4_f32 in 96 cycles instead of 256.  Against float64 the error is smaller than that of the float
// instruction, which rounds after every four k (256 x 4096 outputs, normal operands: 1.0e-7 against 2.1e-7 of a norm at K 1024,
// 1.6e-7 against 4.1e-7 at 4096, 3.1e-7 against 8.1e-7 at 16,384; a whole model's logits 2.6e-6 against 6.4e-6).
// An infinite operand gives NaN (its pieces are inf and NaN), where a float product may give an infinity; pieces
// below a float's smallest normal number may be lost, which is as much below the float they belong to.
//
// The order of an output's sum is the same in every kernel that includes this, so a row of X has the same bits alone
// and among thousands: K is walked in steps of 32, a step is the six products in the order of f3_step below,
// the steps fall into F3_SLICES contiguous slices of ceil(steps / F3_SLICES), each slice is summed from zero and the
// slices' sums are added in ascending order.  Inside a step lane (r, q) of either operand holds row r and
// k = 4 q .. 4 q + 3 and 16 + 4 q .. 16 + 4 q + 3, two 16-byte pieces of a row of floats.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;

#define F3_SLICES 8
#define F3_STEP 32

struct F3Pair {   // two floats' pieces, packed
    uint32_t h, m, l;
};

__device__ __forceinline__ uint32_t f3_round(float a, float b) {
    const bf16x2 v = __builtin_convertvector((f32x2_t){a, b}, bf16x2);
    return __builtin_bit_cast(uint32_t, v);
}

// c minus the first or the second of a pair: the pair's dot product with (-1, 0) or (0, -1) added to c.  One instruction where
// widening the piece and subtracting it are two (3.5 instructions a float in all instead of 5.5); exact, as the difference is.
// (The constants pass through a register: as an operand written into the instruction, -1.0 stood for the other half.)
__device__ __forceinline__ float f3_less(float c, uint32_t pair, uint32_t which) {
    asm("" : "+s"(which));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, which), c, false);
}
#define F3_FIRST 0x0000bf80u
#define F3_SECOND 0xbf800000u

__device__ __forceinline__ F3Pair f3_split2(float a, float b) {
    F3Pair p;
    p.h = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    const float ra = f3_less(a, p.h, F3_FIRST), rb = f3_less(b, p.h, F3_SECOND);
    p.m = f3_round(ra, rb);
    p.l = f3_round(f3_less(ra, p.m, F3_FIRST), f3_less(rb, p.m, F3_SECOND));
    return p;
}

struct F3Frag {   // one lane's part of a fragment of 16 rows x 32 k
    uint4 h, m, l;
};

__device__ __forceinline__ F3Frag f3_split(const float4& lo, const float4& hi) {
    const F3Pair a = f3_split2(lo.x, lo.y), b = f3_split2(lo.z, lo.w), c = f3_split2(hi.x, hi.y), d = f3_split2(hi.z, hi.w);
    F3Frag f;
    f.h = make_uint4(a.h, b.h, c.h, d.h);
    f.m = make_uint4(a.m, b.m, c.m, d.m);
    f.l = make_uint4(a.l, b.l, c.l, d.l);
    return f;
}

// The slot of lane (r, q)'s 16 bytes in a row group's 1 KB of LDS.  A 16-byte read is served for lanes 0-3, 12-15, 20-23 and 24-27 at
// once, then 4-11, 16-19 and 28-31, and so on; an 8-byte write along rows brings four neighbouring rows of all q.  Rows are
// swapped in fours by q so that both fall on distinct banks (by 4 q alone half of LDS's time went into conflicts).
__device__ __forceinline__ int f3_slot(int r, int q) { return q * 16 + (r ^ (4 * ((q >> 1) ^ (3 * (q & 1))))); }

__device__ __forceinline__ f32x4 f3_mfma(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The products of a step in their order: piece of W (0 h, 1 m, 2 l) and piece of X.  The first five, the small ones, are summed from zero
// and join the sum of the h h products by a float addition: the matrix instruction cuts off what lies below its largest
// term's last bits, and five times a step that is a bias (-9e-8 of a mean output at K 4096, against 5e-10 this way).
#define F3_SMALL 5
__device__ __forceinline__ constexpr int f3_w(int p) { return p == 0 ? 2 : p == 2 || p == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int f3_x(int p) { return p == 1 ? 2 : p == 2 || p == 4 ? 1 : 0; }
__device__ __forceinline__ const uint4& f3_piece(const F3Frag& f, int i) { return i == 0 ? f.h : i == 1 ? f.m : f.l; }

// One step of TILES tiles of W (from number t0 of acc on) against one group of X
template <int TILES, int RT, int G>
__device__ __forceinline__ void f3_step(const F3Frag (&w)[TILES], const F3Frag& x, f32x4 (&acc)[RT][G], int t0, int g) {
    f32x4 c[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) c[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < F3_SMALL; ++p)
#pragma unroll
        for (int t = 0; t < TILES; ++t) c[t] = f3_mfma(f3_piece(w[t], f3_w(p)), f3_piece(x, f3_x(p)), c[t]);
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t0 + t][g] = f3_mfma(w[t].h, x.h, acc[t0 + t][g]);
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t0 + t][g] += c[t];
}
