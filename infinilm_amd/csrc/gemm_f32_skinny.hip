// C[M,N] = alpha * (X[M,K] W[N,K]^T + bias) in 32-bit for few rows of X (M <= 64): the projections of a decode step
// on the 32-bit path, bound by reading W once.
//
// The products run on the bfloat16 matrix cores in three pieces a float (f32_split.h), W rows on the A side and tokens on
// the B side.  The eight waves of a workgroup take the eight slices of K and keep DEPTH steps of loads in flight; a load
// instruction takes eight rows' whole 128-byte lines (32 k).  Lanes that gather a fragment from 16 rows, as this kernel had
// it, are taken in at 31 GB/s a compute unit whatever the source, X as slowly as W.  A wave cuts what has arrived into pieces and
// turns it into fragments through LDS of its own: no barrier until the partial tiles meet, in wave order.
// Eight rows, before and after: 6912 x 2304 19.8 -> 14.3 us (4.5 TB/s), 2304 x 5760 23.3 -> 17.7, 122753 x 2304 266 -> 195,
// 32768 x 4096 111 -> 91 (5.9 TB/s); 64 rows 58 -> 28, 69 -> 43, 852 -> 412 and 346 -> 174.
// K must be a multiple of 4 and rows 16-byte aligned.
#include "f32_split.h"

#define FS_WAVES F3_SLICES

// XG: groups of 8 rows of X; RT: tiles of 16 W rows a workgroup; DEPTH: steps of 32 k in flight
template <int XG, int RT, int DEPTH>
__global__ void __launch_bounds__(FS_WAVES * 64, XG <= 2 ? 4 : 2)
gemm_f32_skinny_kernel(float* __restrict__ C, const float* __restrict__ X, const float* __restrict__ W,
                       const float* __restrict__ bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha) {
    constexpr int MG = (XG + 1) / 2;
    struct Frags {
        uint4 at[RT + MG][3][64];   // [tile of W, then group of X][piece][slot]
    };
    union Lds {
        Frags frag[FS_WAVES];
        float part[FS_WAVES][RT][MG][64][4];
    };
    __shared__ Lds lds;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;       // place in a fragment
    const int lrow = lane >> 3, lk4 = lane & 7;   // place in a load: row, 16-byte piece of its line
    const int n0 = blockIdx.x * (16 * RT);
    const int steps_total = (K + F3_STEP - 1) / F3_STEP;
    const int per = (steps_total + F3_SLICES - 1) / F3_SLICES;
    const int s0 = wave * per;
    const int s1 = (s0 + per < steps_total) ? s0 + per : steps_total;
    const int k4_last = (K >> 2) - 1;   // last valid group of 4 elements of a row

    const float4* wp[2 * RT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int row = n0 + 8 * i + lrow;
        wp[i] = reinterpret_cast<const float4*>(W + (size_t)(row < N ? row : N - 1) * ldw);
    }
    const float4* xp[XG];
    bool xok[XG];
#pragma unroll
    for (int i = 0; i < XG; ++i) {
        const int row = 8 * i + lrow;
        xok[i] = row < M;
        xp[i] = reinterpret_cast<const float4*>(X + (size_t)(xok[i] ? row : M - 1) * lda);
    }
    Frags& mine = lds.frag[wave];
    const int get = f3_slot(r, q);
    int put[2];   // in 8 bytes: rows 0 .. 7 and 8 .. 15 of a group
#pragma unroll
    for (int h = 0; h < 2; ++h) put[h] = f3_slot(lrow + 8 * h, lk4 & 3) * 2 + (lk4 >> 2);
    if (XG & 1) {   // the last group's rows 8 .. 15 hold nothing
#pragma unroll
        for (int p = 0; p < 3; ++p) reinterpret_cast<uint2*>(&mine.at[RT + MG - 1][p][0])[put[1]] = make_uint2(0u, 0u);
    }
    f32x4 acc[RT][MG];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int g = 0; g < MG; ++g) acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Unconditional 16-byte loads from clamped addresses, the steps after the slice's end those of its last one again; what
    // lies beyond K, beyond the slice or beyond M is replaced by zeros on the X side.
    float4 a[DEPTH][2 * RT], b[DEPTH][XG];
    auto load = [&](int i, int s) {
        const int k4 = 8 * (s < s1 ? s : s1 - 1) + lk4, k4c = k4 < k4_last ? k4 : k4_last;
#pragma unroll
        for (int t = 0; t < 2 * RT; ++t) a[i][t] = wp[t][k4c];
#pragma unroll
        for (int g = 0; g < XG; ++g) b[i][g] = xp[g][k4c];
    };
    auto cut = [&](int at, int h, const float4& v) {
        const F3Pair c = f3_split2(v.x, v.y), d = f3_split2(v.z, v.w);
        uint2* to = reinterpret_cast<uint2*>(&mine.at[at][0][0]) + put[h];
        to[0] = make_uint2(c.h, d.h);
        to[128] = make_uint2(c.m, d.m);
        to[256] = make_uint2(c.l, d.l);
    };
    auto frag = [&](int at) { return F3Frag{mine.at[at][0][get], mine.at[at][1][get], mine.at[at][2][get]}; };
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    if (s0 < s1) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {   // (in the loop's order: the waits count loads, and take the worse of two orders)
            load(i, s0 + i);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto step = [&](int i, int s, bool more) {
            const bool live = 8 * s + lk4 <= k4_last;
#pragma unroll
            for (int t = 0; t < 2 * RT; ++t) cut(t >> 1, t & 1, a[i][t]);
#pragma unroll
            for (int g = 0; g < XG; ++g) cut(RT + (g >> 1), g & 1, live && xok[g] ? b[i][g] : zero);
            if (more) load(i, s + DEPTH);
            // the wave's own writes before its reads: LDS serves a wave in order, the compiler keeps the order here
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            F3Frag w[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t) w[t] = frag(t);
#pragma unroll
            for (int g = 0; g < MG; ++g) {
                const F3Frag x = frag(RT + g);
                f3_step(w, x, acc, 0, g);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            __builtin_amdgcn_sched_barrier(0);
        };
        int s = s0;
        for (; s + DEPTH < s1; s += DEPTH) {
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) step(i, s + i, true);
        }
#pragma unroll
        for (int i = 0; i < DEPTH; ++i)
            if (s + i < s1) step(i, s + i, false);
    }
    __syncthreads();   // (the partial tiles lie where the fragments lay)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int g = 0; g < MG; ++g) *reinterpret_cast<f32x4*>(&lds.part[wave][t][g][lane][0]) = acc[t][g];
    __syncthreads();
    // acc[t][g][e] of lane (r, q) is output row n0 + t*16 + q*4 + e for token g*16 + r
    for (int idx = threadIdx.x; idx < RT * MG * 64 * 4; idx += FS_WAVES * 64) {
        const int e = idx & 3, l = (idx >> 2) & 63, tg = idx >> 8;
        const int t = tg / MG, g = tg % MG;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < FS_WAVES; ++w) v += lds.part[w][t][g][l][e];
        const int n = n0 + t * 16 + (l >> 4) * 4 + e;
        const int m = g * 16 + (l & 15);
        if (n < N && m < M) {
            if (bias != nullptr) v += bias[n];
            C[(size_t)m * ldc + n] = alpha * v;
        }
    }
}

extern "C" int ilm_gemm_f32_skinny(void* C, const void* X, const void* W, const void* bias, int M, int N, int K,
                                   int lda, int ldw, int ldc, float alpha, hipStream_t stream) {
    ILM_REQUIRE(M > 0 && M <= 64 && N > 0 && K > 0, "gemm_f32_skinny: needs 1 <= M <= 64, got M=%d N=%d K=%d", M, N, K);
    ILM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda >= K && ldw >= K && ldc >= N,
                "gemm_f32_skinny: K=%d lda=%d ldw=%d ldc=%d", K, lda, ldw, ldc);
    ILM_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_f32_skinny: operands must be 16-byte aligned");
#define FS_CASE(XG_, RT_, DEPTH_)                                                                               \
    gemm_f32_skinny_kernel<XG_, RT_, DEPTH_><<<(N + 16 * RT_ - 1) / (16 * RT_), FS_WAVES * 64, 0, stream>>>(    \
        (float*)C, (const float*)X, (const float*)W, (const float*)bias, M, N, K, lda, ldw, ldc, alpha)
    // Two tiles a workgroup, for which X is read and cut once, where one a workgroup would be more than one a compute unit
    // (M 8, K 2304: 14.3 us against 16.7 at N 6912, 11.6 against 9.6 at N 2304; K 4096: 18.5 against 15.9 at N 4096).  Not where
    // X is eight rows and K long: the deeper pipeline of one tile counts more (N 32768, K 4096: 100.6 against 91.2 us).
    const bool tall = N > 16 * ilm_num_cus() && (M > 8 || N < 16384 || K < 4096);
    if (M <= 8) {
        if (tall) FS_CASE(1, 2, 3);
        else FS_CASE(1, 1, 6);
    } else if (M <= 16) {
        if (tall) FS_CASE(2, 2, 2);
        else FS_CASE(2, 1, 4);
    } else if (M <= 32) {
        if (tall) FS_CASE(4, 2, 3);
        else FS_CASE(4, 1, 4);
    } else if (M <= 48) {
        if (tall) FS_CASE(6, 2, 2);
        else FS_CASE(6, 1, 2);
    } else {
        if (tall) FS_CASE(8, 2, 2);
        else FS_CASE(8, 1, 2);
    }
#undef FS_CASE
    ILM_LAUNCH_CHECK("gemm_f32_skinny");
    return 0;
}
