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
//
// Two more forms have the kernel that would follow in their epilogue, for which a workgroup takes two tiles whose outputs belong
// together and the thread that reduces one output reduces its partner: gate and up rows of a feed-forward (SwiGLU), and the
// halves of 16 rotation pairs of a query or key head, with the write into the paged cache.  Bit for bit what the
// two kernels give, without a launch of 4.8 and 5.6 us each, which is what such small kernels take.
#include "f32_split.h"

#define FS_WAVES F3_SLICES
#define FS_PLAIN 0
#define FS_GLU 1
#define FS_ROPE 2

struct FsRope {   // what FS_ROPE's epilogue needs (as gemm_qkv_rope.hip)
    const int* pos;
    const float *cosT, *sinT;
    float *kc, *vc;
    const int* slots;
    int nh, nkv, d, page;
};

// XG: groups of 8 rows of X; RT: tiles of 16 W rows a workgroup; DEPTH: steps of 32 k in flight.  FORM: FS_GLU: N outputs from 2 N
// rows of W; FS_ROPE: C is the queries' rows
template <int XG, int RT, int DEPTH, int FORM>
__global__ void __launch_bounds__(FS_WAVES * 64, XG <= 2 ? 4 : 2)
gemm_f32_skinny_kernel(float* __restrict__ C, const float* __restrict__ X, const float* __restrict__ W,
                       const float* __restrict__ bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int act, FsRope rope) {
    static_assert(FORM == FS_PLAIN || RT == 2, "outputs in pairs");
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
    const int n0 = FORM == FS_ROPE ? (int)(blockIdx.x / (rope.d / 32)) * rope.d + (int)(blockIdx.x % (rope.d / 32)) * 16
                                   : blockIdx.x * (FORM == FS_GLU ? 16 : 16 * RT);
    const int second = FORM == FS_ROPE ? rope.d / 2 : N;   // the partner's row after an output's (FS_GLU, FS_ROPE)
    const int steps_total = (K + F3_STEP - 1) / F3_STEP;
    const int per = (steps_total + F3_SLICES - 1) / F3_SLICES;
    const int s0 = wave * per;
    const int s1 = (s0 + per < steps_total) ? s0 + per : steps_total;
    const int k4_last = (K >> 2) - 1;   // last valid group of 4 elements of a row

    const float4* wp[2 * RT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int in = FORM == FS_PLAIN ? 8 * i : 8 * (i & 1);
        int row = n0 + in + lrow;
        if (FORM != FS_ROPE) row = row < N ? row : N - 1;
        if (FORM != FS_PLAIN && i >= 2) row += second;
        wp[i] = reinterpret_cast<const float4*>(W + (size_t)row * ldw);
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
    if (FORM != FS_PLAIN) {
        for (int idx = threadIdx.x; idx < MG * 64 * 4; idx += FS_WAVES * 64) {
            const int e = idx & 3, l = (idx >> 2) & 63, g = idx >> 8;
            const int n = n0 + (l >> 4) * 4 + e, m = g * 16 + (l & 15);
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int w = 0; w < FS_WAVES; ++w) {
                a += lds.part[w][0][g][l][e];
                b += lds.part[w][RT - 1][g][l][e];
            }
            if (m >= M || (FORM == FS_GLU && n >= N)) continue;
            if (bias != nullptr) {
                a += bias[n];
                b += bias[n + second];
            }
            if (FORM == FS_GLU) {
                C[(size_t)m * ldc + n] = glu_act(a, act) * b;
                continue;
            }
            const int d = rope.d, half = d / 2, hs = n / d, i = n % d, slot = rope.slots != nullptr ? rope.slots[m] : -1;
            if (hs >= rope.nh + rope.nkv) {   // values are cached transposed, [pages, nkv, d, page]
                if (slot < 0) continue;
                float* to = rope.vc + ((size_t)(slot / rope.page) * rope.nkv + (hs - rope.nh - rope.nkv)) * d * rope.page + (slot % rope.page);
                to[(size_t)i * rope.page] = a;
                to[(size_t)(i + half) * rope.page] = b;
                continue;
            }
            const size_t at = (size_t)rope.pos[m] * half + i;
            const float cs = rope.cosT[at], sn = rope.sinT[at];
            const float ra = a * cs - b * sn, rb = b * cs + a * sn;
            float* to;
            if (hs < rope.nh) {
                to = C + (size_t)m * ldc + n;
            } else {
                if (slot < 0) continue;
                to = rope.kc + (((size_t)(slot / rope.page) * rope.nkv + (hs - rope.nh)) * rope.page + (slot % rope.page)) * d + i;
            }
            to[0] = ra;
            to[half] = rb;
        }
        return;
    }
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

#define FS_RUN(XG_, RT_, DEPTH_, FORM_, BLOCKS_)                                                                 \
    gemm_f32_skinny_kernel<XG_, RT_, DEPTH_, FORM_><<<BLOCKS_, FS_WAVES * 64, 0, stream>>>(                      \
        (float*)C, (const float*)X, (const float*)W, (const float*)bias, M, N, K, lda, ldw, ldc, alpha, act, rope)
#define FS_PAIRS(FORM_, BLOCKS_)                                                                                 \
    {                                                                                                            \
        if (M <= 8) FS_RUN(1, 2, 3, FORM_, BLOCKS_);                                                             \
        else if (M <= 16) FS_RUN(2, 2, 2, FORM_, BLOCKS_);                                                       \
        else if (M <= 32) FS_RUN(4, 2, 3, FORM_, BLOCKS_);                                                       \
        else if (M <= 48) FS_RUN(6, 2, 2, FORM_, BLOCKS_);                                                       \
        else FS_RUN(8, 2, 2, FORM_, BLOCKS_);                                                                    \
    }

static int fs_check(const char* name, const void* X, const void* W, int M, int N, int K, int lda, int ldw) {
    ILM_REQUIRE(M > 0 && M <= 64 && N > 0 && K > 0, "%s: needs 1 <= M <= 64, got M=%d N=%d K=%d", name, M, N, K);
    ILM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda >= K && ldw >= K, "%s: K=%d lda=%d ldw=%d", name, K, lda, ldw);
    ILM_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "%s: operands must be 16-byte aligned", name);
    return 0;
}

extern "C" int ilm_gemm_f32_skinny(void* C, const void* X, const void* W, const void* bias, int M, int N, int K,
                                   int lda, int ldw, int ldc, float alpha, hipStream_t stream) {
    if (fs_check("gemm_f32_skinny", X, W, M, N, K, lda, ldw) != 0) return -1;
    ILM_REQUIRE(ldc >= N, "gemm_f32_skinny: N=%d ldc=%d", N, ldc);
    const int act = 0;
    const FsRope rope = {};
    // Two tiles a workgroup, for which X is read and cut once, where one a workgroup would be more than one a compute unit
    // (M 8, K 2304: 14.3 us against 16.7 at N 6912, 11.6 against 9.6 at N 2304; K 4096: 18.5 against 15.9 at N 4096).  Not where
    // X is eight rows and K long: the deeper pipeline of one tile counts more (N 32768, K 4096: 100.6 against 91.2 us).
    const bool tall = N > 16 * ilm_num_cus() && (M > 8 || N < 16384 || K < 4096);
    const int blocks = (N + 15) / 16;
    if (tall) FS_PAIRS(FS_PLAIN, (N + 31) / 32)
    else if (M <= 8) FS_RUN(1, 1, 6, FS_PLAIN, blocks);
    else if (M <= 16) FS_RUN(2, 1, 4, FS_PLAIN, blocks);
    else if (M <= 32) FS_RUN(4, 1, 4, FS_PLAIN, blocks);
    else if (M <= 48) FS_RUN(6, 1, 2, FS_PLAIN, blocks);
    else FS_RUN(8, 1, 2, FS_PLAIN, blocks);
    ILM_LAUNCH_CHECK("gemm_f32_skinny");
    return 0;
}

// C[M, ldc] = act(X Wg^T + bg) * (X Wu^T + bu), W = [Wg; Wu] of I rows each, bias [2 I] or null
extern "C" int ilm_gemm_f32_glu(void* C, const void* X, const void* W, const void* bias, int M, int I, int K,
                                int lda, int ldw, int ldc, int act, hipStream_t stream) {
    if (fs_check("gemm_f32_glu", X, W, M, I, K, lda, ldw) != 0) return -1;
    ILM_REQUIRE(ldc >= I, "gemm_f32_glu: I=%d ldc=%d", I, ldc);
    const float alpha = 1.f;
    const int N = I;
    const FsRope rope = {};
    FS_PAIRS(FS_GLU, (I + 15) / 16)
    ILM_LAUNCH_CHECK("gemm_f32_glu");
    return 0;
}

// C [M, ldc] receives the rotated query heads; k (rotated) and v go to the cache slots (slots may be null: nothing
// is cached).  W [(nh + 2 nkv) d, ldw] holds the q, k, v rows in this order, bias as many numbers or null; all of a head is rotated.
extern "C" int ilm_gemm_f32_rope(void* C, int ldc, const void* X, int lda, const void* W, int ldw, const void* bias, int M, int K,
                                 const void* pos, const void* cosT, const void* sinT, void* kc, void* vc, const void* slots,
                                 int nh, int nkv, int d, int page, hipStream_t stream) {
    ILM_REQUIRE(nh > 0 && nkv >= 0 && d > 0 && d % 32 == 0, "gemm_f32_rope: %d + 2 * %d heads of %d", nh, nkv, d);
    const int N = (nh + 2 * nkv) * d;
    if (fs_check("gemm_f32_rope", X, W, M, N, K, lda, ldw) != 0) return -1;
    ILM_REQUIRE(ldc >= nh * d, "gemm_f32_rope: rows of %d for %d heads of %d", ldc, nh, d);
    ILM_REQUIRE(slots == nullptr || (page > 0 && kc != nullptr && vc != nullptr), "gemm_f32_rope: cache missing");
    const float alpha = 1.f;
    const int act = 0;
    const FsRope rope = {(const int*)pos, (const float*)cosT, (const float*)sinT, (float*)kc, (float*)vc, (const int*)slots, nh, nkv, d, page};
    FS_PAIRS(FS_ROPE, N / 32)
    ILM_LAUNCH_CHECK("gemm_f32_rope");
    return 0;
}
