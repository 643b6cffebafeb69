// bfloat16 products of portions of prompts, C[M,N] = X[M,K] W[N,K]^T (+ bias), where the outputs make about one round of tiles over the
// chip: beyond that the vendor library's tiles win, which keep the matrix cores busier (1.4 PFLOP/s against 1.2 at 2048 x 32768 x
// 4096).  K in steps of 64, whose rows of X and W go from memory into LDS without passing through registers, NS stages deep; the
// second half of a stage is read while the first is multiplied, and the next stage's first half while the second is.
//
// What bounds it: with one tile a compute unit a chain of K / 64 stages (0.28 us each for 128 x 64 outputs, of which the matrix cores are
// busy 0.1), the start and the end.  So tiles are chosen to fill the chip once (kernels.py), stages are as many as LDS holds, and the results
// leave through LDS in whole lines (eight bytes a lane straight from the sums: 2048 x 1024 x 1024 10.9 us, now 9.1; 2048 x 8192 x 1024 49.8, now 34.9).
//
// Three forms: the product alone; act(gate) * up of a feed-forward's first product (the rows of W are taken so that a lane holds gate
// and up of the same outputs); and the fused q | k | v projection with rotation and the write into the paged cache.  us, against the vendor
// library's product (and the kernel after it):
//   product   2048 x 1024 x 1024  9.1 / 10.7, x 4096 22.3 / 25.9; 1000 x 2048 x 2048 13.6 / 16.5; 300 x 1024 x 1024 5.6 / 7.1; 100 x 8192 x 1024 6.5 / 9.8
//   gate, up  2048 x 8192 x 1024 40.0 / 42.5; 1000 rows 23.6 / 27.7; 300 rows 12.6 / 17.4; 100 rows 9.2 / 12.4
//   q, k, v   2048 x 1280 x 1024 18.7 / 20.1; 1000 rows 10.6 / 15.1; 300 rows 7.3 / 10.3; 300 x 4608 x 4096 23.8 / 27.7
// An output's sum runs over K in steps of 32 from the first on, whatever the form and the tile.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) void* lds_ptr;

#define GP_BK 64   // k a stage: a row is one 128-byte line

enum { GP_PLAIN = 0, GP_GLU = 1, GP_ROPE = 2 };

struct GpArgs {
    const bf16* X;
    const bf16* W;
    const bf16* bias;
    bf16* C;
    int M, N, K;        // N: output columns a row of C (GLU: W has 2 N rows)
    int lda, ldw, ldc;
    int m_tiles, n_tiles, group;   // group: m tiles that the n tiles are walked with
    int glu;
    // rope
    const int* pos;
    const float* cosT;
    const float* sinT;
    bf16* kc;
    bf16* vc;
    const int* slots;
    int nh, nkv, d, page;
};

__device__ __forceinline__ f32x4 gp_mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The row of W that stands at place j of tile nt
template <int BN, int WN, int EPI>
__device__ __forceinline__ int gp_w_row(const GpArgs& A, int nt, int j) {
    if (EPI == GP_PLAIN) {
        const int n = nt * BN + j;
        return n < A.N ? n : A.N - 1;
    }
    const int seg = j / WN, jj = j % WN, second = jj / (WN / 2), p = nt * (BN / 2) + seg * (WN / 2) + jj % (WN / 2);
    if (EPI == GP_GLU) return (p < A.N ? p : A.N - 1) + second * A.N;
    const int half = A.d / 2, pairs = A.N / 2, pc = p < pairs ? p : pairs - 1;
    return pc / half * A.d + pc % half + second * half;
}

// BAND: the tiles are walked in bands of `group` m tiles (gp_group); else all m tiles of an n tile one after the other
template <int BM, int BN, int WM, int WN, int NS, int EPI, bool BAND>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64, 2)
gemm_portion_kernel(const GpArgs A) {
    constexpr int NW = (BM / WM) * (BN / WN), ROWS = BM + BN, GROUPS = ROWS / 8, PER = GROUPS / NW, TM = WM / 16, TN = WN / 16;
    static_assert(GROUPS % NW == 0 && (BN / 8) % NW == 0, "whole loads");
    constexpr int OUT = EPI == GP_GLU ? BN / 2 : BN, PITCH = OUT + 8;   // columns a tile gives, elements between its rows in LDS
    constexpr int STAGES = NS * ROWS * GP_BK, STAGED = BM * PITCH;
    __shared__ __align__(16) bf16 lds[STAGES > STAGED ? STAGES : STAGED];   // [stage][rows of W, then rows of X][64]; at the end the tile's results
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, q = lane >> 4;
    int mt, nt;
    {
        const int total = A.m_tiles * A.n_tiles, per = total >> 3, rem = total & 7, xcd = blockIdx.x & 7;
        const int id = xcd * per + (xcd < rem ? xcd : rem) + ((int)blockIdx.x >> 3);
        int first = 0, rows = A.m_tiles;
        if (BAND) {
            first = id / (A.group * A.n_tiles) * A.group;
            rows = A.m_tiles - first < A.group ? A.m_tiles - first : A.group;
        }
        const int at = id - first * A.n_tiles;
        mt = first + at % rows;
        nt = at / rows;
    }
    const int m0 = mt * BM;
    const int wn = wave % (BN / WN), wm = wave / (BN / WN);

    const int lrow = lane >> 3, piece = (lane & 7) ^ lrow;
    uint32_t from[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int row = (wave + NW * i) * 8 + lrow;
        if (NW * i < BN / 8) {
            from[i] = (uint32_t)gp_w_row<BN, WN, EPI>(A, nt, row) * ((uint32_t)A.ldw * 2u) + piece * 16;
        } else {
            const int m = m0 + row - BN;
            from[i] = (uint32_t)(m < A.M ? m : A.M - 1) * ((uint32_t)A.lda * 2u) + piece * 16;
        }
    }
    const char* wb = reinterpret_cast<const char*>(A.W);
    const char* xb = reinterpret_cast<const char*>(A.X);
    // (The compiler waits for all loads into LDS before it reads any of it, so these are written out and waited for by number.  They have no
    // register to deliver to.)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)(&lds[0]) + (uint32_t)wave * 1024;
    auto issue = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + (uint32_t)(buf * ROWS * 128 + NW * i * 1024)),
                         "v"(from[i]), "s"(NW * i < BN / 8 ? wb : xb)
                         : "m0", "memory");
        wb += GP_BK * 2;
        xb += GP_BK * 2;
    };
    // The lane's outputs' biases, asked for ahead of the stages: behind them their way through memory cost 0.8 to 1.9 us (65 x 1024 x 1024
    // 6.2 us, now 5.5, as without a bias and as the library's product with its addend; 2048 x 2048 x 1536 19.8, now 16.3, library 17.6).  With tiles
    // of 256 x 256, whose sums leave no registers for them, right after the stages.
    constexpr bool EARLY = TM * TN <= 16;
    bf16 bs[TN][4];
    auto load_bias = [&]() {
        if (A.bias == nullptr) return;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int tt = t % (TN / 2), second = t / (TN / 2);   // (gate, up and pairs: the second half of the t are the other of the same outputs)
            int n;
            if (EPI == GP_ROPE) {
                const int half = A.d / 2, pairs = A.N / 2, p = nt * (BN / 2) + wn * (WN / 2) + tt * 16 + 4 * q, pc = p < pairs ? p : 0;
                n = pc / half * A.d + pc % half + second * half;
            } else {
                n = EPI == GP_GLU ? nt * OUT + wn * (WN / 2) + tt * 16 + 4 * q : nt * OUT + wn * WN + t * 16 + 4 * q;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int at = EPI == GP_ROPE ? n + e : n + e < A.N ? n + e : A.N - 1;
                bs[t][e] = A.bias[EPI == GP_GLU ? at + second * A.N : at];
            }
        }
    };
    if (EARLY) load_bias();
    auto biased = [&](float v, int t, int e) { return A.bias != nullptr ? v + to_f32(bs[t][e]) : v; };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int g = 0; g < TM; ++g) acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int stages = A.K / GP_BK;
    const int sw = r & 7;
    uint4 a[2][TN], b[2][TM];
    auto read = [&](int s, int buf) {
        const uint4* base = reinterpret_cast<const uint4*>(&lds[0]) + buf * (ROWS * 8) + ((s * 4 + q) ^ sw);
        const uint4* ws = base + (wn * WN + r) * 8;
        const uint4* xs = base + (BN + wm * WM + r) * 8;
#pragma unroll
        for (int t = 0; t < TN; ++t) a[s][t] = ws[t * 128];
#pragma unroll
        for (int g = 0; g < TM; ++g) b[s][g] = xs[g * 128];
    };
    auto multiply = [&](int s) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < TM; ++g)
#pragma unroll
            for (int t = 0; t < TN; ++t) acc[t][g] = gp_mfma(a[s][t], b[s][g], acc[t][g]);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int ahead = stages < NS ? stages : NS;
    for (int i = 0; i < ahead; ++i) issue(i);
    if (stages > NS - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    int buf = 0, st = 0;
    for (; st + NS < stages; ++st) {
        read(1, buf);
        multiply(0);
        // stage st + 1 has landed (this wave's part), and this wave is done with stage st's buffer
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * PER) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(buf);
        buf = buf + 1 == NS ? 0 : buf + 1;
        read(0, buf);
        multiply(1);
    }
    for (; st + 1 < stages; ++st) {
        read(1, buf);
        multiply(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        buf = buf + 1 == NS ? 0 : buf + 1;
        read(0, buf);
        multiply(1);
    }
    read(1, buf);
    multiply(0);
    multiply(1);
    if (!EARLY) load_bias();
    // acc[t][g][e] of lane (r, q): row wm WM + 16 g + r of the tile, place wn WN + 16 t + 4 q + e
    if (EPI == GP_ROPE) {
        // (values go straight into their transposed cache; queries and keys through LDS, first halves of pairs ahead of second halves)
        const int half = A.d / 2, pairs = A.N / 2;
        __syncthreads();
#pragma unroll
        for (int g = 0; g < TM; ++g) {
            const int row = wm * WM + g * 16 + r, m = m0 + row < A.M ? m0 + row : A.M - 1;
            const int p_m = A.pos[m], slot = A.slots != nullptr && m0 + row < A.M ? A.slots[m] : -1;
#pragma unroll
            for (int t = 0; t < TN / 2; ++t) {
                const int place = wn * (WN / 2) + t * 16 + 4 * q, pair = nt * (BN / 2) + place;   // (16 pairs from a multiple of 16 on: one head's)
                if (pair >= pairs) continue;
                const int hs = pair / half, i0 = pair % half;
                float v[2][4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int h = 0; h < 2; ++h) v[h][e] = to_f32(from_f32<bf16>(biased(acc[t + h * (TN / 2)][g][e], t + h * (TN / 2), e)));
                if (hs >= A.nh + A.nkv) {
                    if (slot < 0) continue;
                    bf16* dst = A.vc + ((size_t)(slot / A.page) * A.nkv + (hs - A.nh - A.nkv)) * A.d * A.page + (slot % A.page);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        dst[(size_t)(i0 + e) * A.page] = from_f32<bf16>(v[0][e]);
                        dst[(size_t)(i0 + half + e) * A.page] = from_f32<bf16>(v[1][e]);
                    }
                    continue;
                }
                const float4 cs = *reinterpret_cast<const float4*>(A.cosT + (size_t)p_m * half + i0);
                const float4 sn = *reinterpret_cast<const float4*>(A.sinT + (size_t)p_m * half + i0);
                const float c4[4] = {cs.x, cs.y, cs.z, cs.w}, s4[4] = {sn.x, sn.y, sn.z, sn.w};
                bf16 o[2][4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[0][e] = from_f32<bf16>(v[0][e] * c4[e] - v[1][e] * s4[e]);
                    o[1][e] = from_f32<bf16>(v[1][e] * c4[e] + v[0][e] * s4[e]);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) *reinterpret_cast<uint2*>(&lds[row * PITCH + h * (BN / 2) + place]) = *reinterpret_cast<const uint2*>(o[h]);
            }
        }
        __syncthreads();
        constexpr int P8 = BN / 8;
        for (int i = tid; i < BM * P8; i += NW * 64) {   // (eight pairs from a multiple of eight on are one head's)
            const int row = i / P8, m = m0 + row, h = i % P8 / (P8 / 2), place = i % (P8 / 2) * 8, pair = nt * (BN / 2) + place;
            if (m >= A.M) break;
            const int hs = pair / half, at = pair % half + h * half;
            if (pair >= pairs || hs >= A.nh + A.nkv) continue;
            bf16* dst = A.C + (size_t)m * A.ldc + (size_t)hs * A.d + at;
            if (hs >= A.nh) {
                const int slot = A.slots != nullptr ? A.slots[m] : -1;
                if (slot < 0) continue;
                dst = A.kc + (((size_t)(slot / A.page) * A.nkv + (hs - A.nh)) * A.page + (slot % A.page)) * A.d + at;
            }
            *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(&lds[row * PITCH + h * (BN / 2) + place]);
        }
        return;
    }
    // The results go to memory through LDS, whole lines of a row at a time
    __syncthreads();
#pragma unroll
    for (int g = 0; g < TM; ++g) {
        const int row = wm * WM + g * 16 + r;
#pragma unroll
        for (int t = 0; t < (EPI == GP_GLU ? TN / 2 : TN); ++t) {
            const int col = wn * (EPI == GP_GLU ? WN / 2 : WN) + t * 16 + 4 * q;
            bf16 o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (EPI == GP_GLU) {
                    const float vg = biased(acc[t][g][e], t, e), vu = biased(acc[t + TN / 2][g][e], t + TN / 2, e);
                    // (gate and up rounded to bfloat16 first, as the product's kernel alone stores them)
                    o[e] = from_f32<bf16>(glu_act(to_f32(from_f32<bf16>(vg)), A.glu) * to_f32(from_f32<bf16>(vu)));
                } else {
                    o[e] = from_f32<bf16>(biased(acc[t][g][e], t, e));
                }
            }
            *reinterpret_cast<uint2*>(&lds[row * PITCH + col]) = *reinterpret_cast<const uint2*>(o);
        }
    }
    __syncthreads();
    constexpr int P8 = OUT / 8;   // 16-byte pieces a row
    const bool vec = (A.ldc & 7) == 0 && ((uintptr_t)A.C & 15) == 0;
#pragma unroll 4
    for (int i = tid; i < BM * P8; i += NW * 64) {
        const int row = i / P8, m = m0 + row, n = nt * OUT + i % P8 * 8;
        if (m >= A.M) break;
        const bf16* from = &lds[row * PITCH + i % P8 * 8];
        bf16* dst = A.C + (size_t)m * A.ldc + n;
        if (vec && n + 7 < A.N) {
            *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(from);
        } else {
            for (int e = 0; e < 8; ++e)
                if (n + e < A.N) dst[e] = from[e];
        }
    }
}

// M tiles that are walked together before the next n tile.  An XCD takes an eighth of the tiles, consecutive ones, and fetches their rows of X and W into
// its own L2: with all m tiles together all of X for each (2048 x 1024 x 4096 in tiles of 128 x 64: 134 MB in all, 67 MB where four m tiles are
// walked with eight n tiles: 24.1 -> 22.4 us; 1000 x 1024 x 4096 15.2 -> 14.6).  But then a row of W is fetched by several: only where at most two
// thirds of the rows are left (1000 x 2304 x 2304, four fifths, 18.0 -> 18.8), and not for q, k and v (2048 x 1280 x 1024, a round and a
// quarter, in a model's step 16.1 -> 17.6).  Kernels of their own: with the band's two divisions and the arguments they wait for every workgroup starts
// later, and what has no bands loses (985 x 4096 x 4096 36.8 us, 38.3 so; 600 x 4096 x 2048 18.1 and 19.0).
static int gp_group(int m_tiles, int n_tiles, int bm, int bn) {
    const long long per = ((long long)m_tiles * n_tiles + 7) / 8;
    auto rows = [&](int g) { return (long long)g * bm + (per + g - 1) / g * bn; };
    int best = m_tiles;
    for (int g = 1; g < m_tiles && (long long)(g - 1) * bm < rows(best); ++g)
        if (rows(g) < rows(best)) best = g;
    return 3 * rows(best) <= 2 * rows(m_tiles) ? best : m_tiles;
}

// tile: 1: 64 x 64 outputs (gate, up: 64 x 128 rows of W), 2: 128 x 64, 3: 128 x 128, 4: 256 x 128, 5: 256 x 256
#define GP_RUN(BM_, BN_, WM_, WN_, NS_, EPI_, NCOLS_)                                                       \
    {                                                                                                       \
        a.m_tiles = (a.M + BM_ - 1) / BM_;                                                                  \
        a.n_tiles = ((NCOLS_) + BN_ - 1) / BN_;                                                             \
        ILM_REQUIRE((long long)a.m_tiles * a.n_tiles < (1ll << 31), "gemm_portion: too many tiles");        \
        a.group = EPI_ == GP_PLAIN ? gp_group(a.m_tiles, a.n_tiles, BM_, BN_) : a.m_tiles;                  \
        const int threads = (BM_ / WM_) * (BN_ / WN_) * 64;                                                 \
        if (EPI_ == GP_PLAIN && a.group < a.m_tiles)                                                        \
            gemm_portion_kernel<BM_, BN_, WM_, WN_, NS_, EPI_, EPI_ == GP_PLAIN>                            \
                <<<a.m_tiles * a.n_tiles, threads, 0, stream>>>(a);                                         \
        else                                                                                                \
            gemm_portion_kernel<BM_, BN_, WM_, WN_, NS_, EPI_, false>                                       \
                <<<a.m_tiles * a.n_tiles, threads, 0, stream>>>(a);                                         \
    }

static int gp_check(const char* what, int M, int rows, int K, const void* X, int lda, const void* W, int ldw) {
    ILM_REQUIRE(M > 0 && rows > 0 && K > 0 && K % GP_BK == 0, "%s: bad sizes M=%d rows of W=%d K=%d (K in steps of 64)", what, M, rows, K);
    ILM_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K, "%s: K=%d lda=%d ldw=%d", what, K, lda, ldw);
    ILM_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "%s: operands must be 16-byte aligned", what);
    // (a row's place is 32 bits of bytes)
    ILM_REQUIRE((long long)M * lda < (1ll << 31) && (long long)rows * ldw < (1ll << 31), "%s: operands beyond 4 GiB", what);
    return 0;
}

// C [M, ldc] = X W^T + bias (`glu` < 0: W has N rows), or act(X Wg^T + bg) * (X Wu^T + bu), W = [Wg; Wu] of 2 N rows, `glu` the gate's activation
extern "C" int ilm_gemm_portion(void* C, int ldc, const void* X, int lda, const void* W, int ldw, const void* bias, int M, int N, int K,
                                int glu, int tile, hipStream_t stream) {
    if (gp_check("gemm_portion", M, glu < 0 ? N : 2 * N, K, X, lda, W, ldw)) return -1;
    ILM_REQUIRE(ldc >= N && N < (1 << 30), "gemm_portion: N=%d ldc=%d", N, ldc);
    GpArgs a = {};
    a.X = (const bf16*)X; a.W = (const bf16*)W; a.bias = (const bf16*)bias; a.C = (bf16*)C;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldw = ldw; a.ldc = ldc; a.glu = glu;
    if (glu < 0) {
        ILM_REQUIRE(tile >= 1 && tile <= 3, "gemm_portion: there is no tile %d", tile);
        // (128 x 64: one workgroup a unit by the rule, so five stages; three, 2048 x 1024 x 4096 22.9 us, now 22.3; in a model's step 30 -> 27)
        if (tile == 1) GP_RUN(64, 64, 32, 32, 4, GP_PLAIN, N)
        else if (tile == 2) GP_RUN(128, 64, 32, 32, 5, GP_PLAIN, N)
        else GP_RUN(128, 128, 64, 32, 4, GP_PLAIN, N)
    } else {
        ILM_REQUIRE(tile == 1 || tile == 4 || tile == 5, "gemm_portion: there is no tile %d", tile);
        // (beyond two a unit two stages instead of three, so that three share one: 700 x 6144 x 1024, 528 tiles, 18.7 -> 15.3 us, 700 x 8192 x 1024, 704,
        // 18.9 -> 17.1; up to two a unit the third stage is worth more: 700 x 4096 x 768, 352, 10.8 / 11.2, 37 x 8192 x 1024 8.7 / 11.5)
        if (tile == 1 && (long long)((M + 63) / 64) * ((N + 63) / 64) > 2 * ilm_num_cus()) GP_RUN(64, 128, 32, 64, 2, GP_GLU, 2 * N)
        else if (tile == 1) GP_RUN(64, 128, 32, 64, 3, GP_GLU, 2 * N)
        else if (tile == 4) GP_RUN(256, 128, 64, 64, 3, GP_GLU, 2 * N)
        else GP_RUN(256, 256, 128, 64, 2, GP_GLU, 2 * N)
    }
    ILM_LAUNCH_CHECK("gemm_portion");
    return 0;
}

// Q [M, ldq] receives the rotated query heads; k (rotated) and v go to the cache slots (slots may be
// null: nothing is cached; a slot below 0: that token is not).  W [(nh + 2 nkv) d, ldw] holds the q, k, v rows in this order.
extern "C" int ilm_gemm_portion_rope(void* Q, int ldq, const void* X, int lda, const void* W, int ldw, const void* bias,
                                     int M, int K, const void* pos, const void* cosT, const void* sinT, void* kc, void* vc,
                                     const void* slots, int nh, int nkv, int d, int page, int tile, hipStream_t stream) {
    ILM_REQUIRE(nh > 0 && nkv >= 0 && d > 0 && d % 32 == 0 && (long long)(nh + 2 * nkv) * d < (1 << 30),
                "gemm_portion_rope: %d + 2 x %d heads of %d", nh, nkv, d);
    if (gp_check("gemm_portion_rope", M, (nh + 2 * nkv) * d, K, X, lda, W, ldw)) return -1;
    ILM_REQUIRE(ldq >= nh * d && ldq % 8 == 0 && ((uintptr_t)Q & 15) == 0, "gemm_portion_rope: ldq=%d", ldq);
    ILM_REQUIRE(pos != nullptr && ((uintptr_t)cosT & 15) == 0 && ((uintptr_t)sinT & 15) == 0, "gemm_portion_rope: tables must be 16-byte aligned");
    ILM_REQUIRE(slots == nullptr || (page > 0 && kc != nullptr && vc != nullptr && ((uintptr_t)kc & 15) == 0), "gemm_portion_rope: cache missing");
    ILM_REQUIRE(tile == 1 || tile == 2, "gemm_portion_rope: there is no tile %d", tile);
    GpArgs a = {};
    a.X = (const bf16*)X; a.W = (const bf16*)W; a.bias = (const bf16*)bias; a.C = (bf16*)Q;
    a.M = M; a.N = (nh + 2 * nkv) * d; a.K = K; a.lda = lda; a.ldw = ldw; a.ldc = ldq;
    a.pos = (const int*)pos; a.cosT = (const float*)cosT; a.sinT = (const float*)sinT; a.kc = (bf16*)kc; a.vc = (bf16*)vc;
    a.slots = (const int*)slots; a.nh = nh; a.nkv = nkv; a.d = d; a.page = page;
    if (tile == 1) GP_RUN(64, 64, 32, 32, 4, GP_ROPE, a.N)
    else GP_RUN(128, 64, 32, 32, 3, GP_ROPE, a.N)
    ILM_LAUNCH_CHECK("gemm_portion_rope");
    return 0;
}
