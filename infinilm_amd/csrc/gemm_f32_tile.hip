// C[M,N] = alpha * (X[M,K] W[N,K]^T + bias) in 32-bit for many rows of X (portions of prompts on the
// 32-bit path), on the bfloat16 matrix cores in three pieces a float (f32_split.h), which also fixes the order of
// every sum: a row of X has the same bits here as in the few-rows kernel (gemm_f32_skinny.hip), whatever the tile.
//
// What bounds it: six matrix instructions of 16 cycles for 16 x 16 x 32, beside which the vector units cut the operands
// into pieces (5.5 instructions a float, once a workgroup: the larger the tile, the fewer) and LDS passes 6 bytes a float.
// So a tile of 128 x 256 with 64 x 64 outputs a wave where there are enough of them for the chip, smaller ones
// else.  The pieces of two stages of 32 k lie in LDS (147 KB), in fragment order.  Half of the waves cut
// the next stage before they multiply, the other half after: two waves share a SIMD, and one's vector work
// runs beside the other's matrix work.  2,048 rows against the kernel on v_mfma_f32_16x16x4_f32 that this one replaced (tiles of
// 128 x 128, 106 TFLOP/s at most): 32768 x 4096 2.86 ms against 5.20 (192 TFLOP/s, of which the matrix cores are busy half
// the time), 4096 x 16384 1.42 against 2.67, 1024 x 1024 44 us against 106; 300 x 4608 x 4096 142 us against 416.
// K must be a multiple of 4 and rows 16-byte aligned.
#include "f32_split.h"

// BM x BN outputs a workgroup (rows of X, rows of W), WM x WN a wave
template <int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64)
gemm_f32_tile_kernel(float* __restrict__ C, const float* __restrict__ X, const float* __restrict__ W,
                     const float* __restrict__ bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha,
                     int m_tiles, int n_tiles, int vec_store) {
    constexpr int NW = (BM / WM) * (BN / WN), NT = NW * 64, ROWS = BM + BN;
    constexpr int LOADS = ROWS * 8 / NT, W_LOADS = BN * 8 / NT, TM = WM / 16, TN = WN / 16;
    static_assert(ROWS * 8 % NT == 0 && BN * 8 % NT == 0, "whole loads");
    // [stage][group of 16 rows (of W, then of X)][piece][slot]
    __shared__ __align__(16) uint4 lds[2][ROWS / 16][3][64];
    // Workgroups go to the 8 XCDs round-robin: those of one XCD take the m tiles of one n tile one after the
    // other, so a tile of W is fetched into one L2 only.
    int mt, nt;
    {
        const int id = blockIdx.x;
        const int full = (n_tiles / 8) * 8 * m_tiles;   // n tiles in whole rounds of 8
        if (id < full) {
            const int xcd = id & 7, local = id >> 3;
            mt = local % m_tiles;
            nt = (local / m_tiles) * 8 + xcd;
        } else {
            const int rest = id - full;
            mt = rest % m_tiles;
            nt = (n_tiles / 8) * 8 + rest / m_tiles;
        }
    }
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int n0 = nt * BN, m0 = mt * BM;
    const int wn = (wave % (BN / WN)) * TN, wm = BN / 16 + (wave / (BN / WN)) * TM;   // the wave's first row groups
    const bool early = wave < NW / 2;

    const int stages = (K + F3_STEP - 1) / F3_STEP;
    const int per = (stages + F3_SLICES - 1) / F3_SLICES;
    const int k4_last = (K >> 2) - 1;

    // a thread stages 16 bytes (piece tid % 8 of a row's 128) of LOADS rows: tid / 8 + i * NT / 8
    const int lrow = tid >> 3, lk4 = tid & 7;
    const float4* wsrc = reinterpret_cast<const float4*>(W + (size_t)n0 * ldw);
    const float4* xsrc = reinterpret_cast<const float4*>(X + (size_t)m0 * lda);
    // (in 16 bytes: a row of the tile, the tile's last row inside the matrix; rows beyond are that one again)
    const uint32_t w4 = ldw >> 2, x4 = lda >> 2;
    uint32_t wfrom = lrow * w4, xfrom = lrow * x4;
    const uint32_t wlast = (uint32_t)min(N - 1 - n0, BN - 1) * w4, xlast = (uint32_t)min(M - 1 - m0, BM - 1) * x4;
    const int put = (lrow >> 4) * 384 + f3_slot(lrow & 15, lk4 & 3) * 2 + (lk4 >> 2);   // in 8 bytes
    const int get = f3_slot(r, q);
    float4 reg[LOADS];
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    auto fetch = [&](int st) {
        const int k4 = st * 8 + lk4, k4c = k4 < k4_last ? k4 : k4_last;
        asm volatile("" : "+v"(wfrom), "+v"(xfrom));   // the rows' offsets are made here each time: outside the loop they would take LOADS registers
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) reg[i] = wsrc[min(wfrom + i * (NT / 8) * w4, wlast) + (uint32_t)k4c];
#pragma unroll
        for (int i = W_LOADS; i < LOADS; ++i) reg[i] = xsrc[min(xfrom + (i - W_LOADS) * (NT / 8) * x4, xlast) + (uint32_t)k4c];
    };
    auto store = [&](int st) {   // cuts what was fetched for stage st into pieces
        const bool beyond = st * 8 + lk4 > k4_last;   // zeros on the X side, as the few-rows kernel has them
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const float4 v = i >= W_LOADS && beyond ? zero : reg[i];
            const F3Pair a = f3_split2(v.x, v.y), b = f3_split2(v.z, v.w);
            uint2* to = reinterpret_cast<uint2*>(&lds[st & 1][i * (NT / 128)][0][0]) + put;
            to[0] = make_uint2(a.h, b.h);
            to[128] = make_uint2(a.m, b.m);
            to[256] = make_uint2(a.l, b.l);
        }
    };

    f32x4 acc[TN][TM], total[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int g = 0; g < TM; ++g) {
            acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
            total[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    fetch(0);
    store(0);
    fetch(1);
    __syncthreads();
    int in_slice = 0;
    for (int st = 0; st < stages; ++st) {
        if (early && st + 1 < stages) {
            store(st + 1);
            fetch(st + 2);
        }
        if (in_slice == per) {   // a slice ends: its sum joins the total, the next starts from zero
            in_slice = 0;
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int g = 0; g < TM; ++g) {
                    total[t][g] += acc[t][g];
                    acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        ++in_slice;
        // two tiles of W at a time: all of a wave's W fragments would take the registers that its sums need (LDS has room
        // for the second reading of X)
#pragma unroll
        for (int t0 = 0; t0 < TN; t0 += 2) {
            asm volatile("" ::: "memory");   // (X's fragments are read again, not kept)
            F3Frag a[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint4(*at)[64] = lds[st & 1][wn + t0 + t];
                a[t] = F3Frag{at[0][get], at[1][get], at[2][get]};
            }
#pragma unroll
            for (int g = 0; g < TM; ++g) {
                const uint4(*at)[64] = lds[st & 1][wm + g];
                const F3Frag b = F3Frag{at[0][get], at[1][get], at[2][get]};
                f3_step(a, b, acc, t0, g);
            }
        }
        if (!early && st + 1 < stages) {
            store(st + 1);
            fetch(st + 2);
        }
        __syncthreads();
    }
    // acc[t][g][e] of lane (r, q): output row m0 + 16 (wm's group + g) + r, column n0 + 16 (wn + t) + 4 q + e
#pragma unroll
    for (int g = 0; g < TM; ++g) {
        const int m = m0 + (wm - BN / 16 + g) * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int n = n0 + (wn + t) * 16 + 4 * q;
            if (n >= N) continue;
            f32x4 v = total[t][g] + acc[t][g];
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = v[e];
                if (bias != nullptr && n + e < N) x += bias[n + e];
                o[e] = alpha * x;
            }
            float* dst = C + (size_t)m * ldc + n;
            if (vec_store && n + 3 < N) {
                *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) dst[e] = o[e];
            }
        }
    }
}

// `tile`: 0 the rule below, 1 .. 3 one of the three shapes (for measurements and tests)
extern "C" int ilm_gemm_f32_tile(void* C, const void* X, const void* W, const void* bias, int M, int N, int K,
                                 int lda, int ldw, int ldc, float alpha, int tile, hipStream_t stream) {
    ILM_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32_tile: bad sizes M=%d N=%d K=%d", M, N, K);
    ILM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda >= K && ldw >= K && ldc >= N,
                "gemm_f32_tile: K=%d lda=%d ldw=%d ldc=%d", K, lda, ldw, ldc);
    ILM_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_f32_tile: operands must be 16-byte aligned");
    ILM_REQUIRE(lda < (1 << 24) && ldw < (1 << 24), "gemm_f32_tile: rows of %d and %d floats", lda, ldw);   // (offsets inside a tile take 32 bits)
    ILM_REQUIRE(tile >= 0 && tile <= 3, "gemm_f32_tile: there is no tile %d", tile);
    const int vec_store = (ldc % 4 == 0 && ((uintptr_t)C & 15) == 0) ? 1 : 0;
#define FT_RUN(BM_, BN_, WM_, WN_)                                                                                          \
    {                                                                                                                       \
        const int m_tiles = (M + BM_ - 1) / BM_, n_tiles = (N + BN_ - 1) / BN_;                                             \
        ILM_REQUIRE((long long)m_tiles * n_tiles < (1ll << 31), "gemm_f32_tile: too many tiles");                           \
        gemm_f32_tile_kernel<BM_, BN_, WM_, WN_><<<m_tiles * n_tiles, (BM_ / WM_) * (BN_ / WN_) * 64, 0, stream>>>(         \
            (float*)C, (const float*)X, (const float*)W, (const float*)bias, M, N, K, lda, ldw, ldc, alpha, m_tiles,        \
            n_tiles, vec_store);                                                                                            \
    }
    if (tile == 0) {
        // The tile that ends soonest, by what a round of each takes (us at K 4096, measured on 256 units: the ratios count).  128 x
        // 256 and 128 x 128 run one a unit, 325 and 197 a round; of 64 x 64 three share a unit: 95 alone, 142 two of them,
        // 66 each when many follow one another.  2048 x 4096 outputs: 368, 405 and 529 us; 300 x 4608: 324, 197 and 142.
        const long long cus = ilm_num_cus();
        auto count = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
        const long long t1 = 325 * ((count(128, 256) + cus - 1) / cus), t2 = 197 * ((count(128, 128) + cus - 1) / cus);
        const long long n3 = count(64, 64), t3 = n3 <= cus ? 95 : n3 <= 2 * cus ? 142 : 66 * n3 / cus + 10;
        tile = t1 <= t2 && t1 <= t3 ? 1 : t2 <= t3 ? 2 : 3;
    }
    if (tile == 1) FT_RUN(128, 256, 64, 64)
    else if (tile == 2) FT_RUN(128, 128, 64, 32)
    else FT_RUN(64, 64, 32, 32)
#undef FT_RUN
    ILM_LAUNCH_CHECK("gemm_f32_tile");
    return 0;
}
