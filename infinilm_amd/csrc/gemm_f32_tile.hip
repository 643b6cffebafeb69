// C[M,N] = alpha * (X[M,K] W[N,K]^T + bias) in 32-bit for many rows of X (portions of prompts on the
// 32-bit path), on the bfloat16 matrix cores in three pieces a float (f32_split.h), which also fixes the order of
// every sum: a row of X has the same bits here as in the few-rows kernel (gemm_f32_skinny.hip), whatever the tile.
//
// What bounds it: six matrix instructions of 16 cycles for 16 x 16 x 32, beside which the vector units cut the operands
// into pieces (3.5 instructions a float, once a workgroup: the larger the tile, the fewer) and LDS passes 6 bytes a float.
// So a tile of 128 x 256 with 64 x 64 outputs a wave where there are enough of them for the chip, smaller ones
// else.  The pieces of two stages of 32 k lie in LDS (147 KB), in fragment order.  Half of the waves cut
// the next stage before they multiply, the other half after: two waves share a SIMD, and one's vector work
// runs beside the other's matrix work (the one that multiplies goes ahead, s_setprio: 2048 x 4608 x 4096 405 -> 395 us, 4096 x 16384 1,380 -> 1,340,
// 32768 x 4096 2,795 -> 2,760).  2,048 rows against the kernel on v_mfma_f32_16x16x4_f32 that this one replaced (tiles of
// 128 x 128, 106 TFLOP/s at most): 32768 x 4096 2.86 ms against 5.20 (192 TFLOP/s, of which the matrix cores are busy half
// the time), 4096 x 16384 1.42 against 2.67, 1024 x 1024 44 us against 106; 300 x 4608 x 4096 142 us against 416.
// Tiles beyond whole rounds over the chip left most of it idle (288 tiles of 2048 x 4608 on 256 units: two rounds, the second an eighth full;
// 300 x 4608 54 tiles): their eight slices of K go to as many workgroups, and a second kernel adds the slices' sums, 128 KB each, in their
// order.  us, the best whole form and now: 2048 x 4608 x 4096 556 / 396, 300 x 4608 x 4096 142 / 98, 100 x 4096 x 16384 387 / 160, 2048 x 1024
// x 4096 159 / 107, 1024 x 2304 x 5760 260 / 177.
// K must be a multiple of 4 and rows 16-byte aligned.
#include "f32_split.h"


// Tiles whose K is cut: those from number `first` on, `slices` slices of K each, which `parts` workgroups a tile share.  Every slice's
// sum leaves for a workspace and gemm_f32_sum_kernel adds them in their order, so the bits are those of a whole tile.
struct FtCut {
    int first, slices, parts;
};

// Workgroups go to the 8 XCDs round-robin: those of one XCD take the m tiles of one n tile one after the
// other, so a tile of W is fetched into one L2 only.
__device__ __forceinline__ void ft_place(int id, int m_tiles, int n_tiles, int& mt, int& nt) {
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

// BM x BN outputs a workgroup (rows of X, rows of W), WM x WN a wave.  CUT: some slices, whose sums leave one by one.
// GLU: W = [gate; up] of N outputs each, a tile's groups of 16 rows in turn from either, so that a lane holds gate and up of the same outputs and
// writes act(gate) * up, the bits of the product and the activation kernel one after the other, which write the sums (268 MB for 2048 x 32768) and
// read them again.  us, apart / here: 2048 x 32768 x 4096 3,000 / 2,880, 2048 x 8192 x 1024 216 / 199, 1024 x 11520 x 2304 324 / 312, in cut tiles 1300 x
// 32768 x 4096 2,046 / 1,982, 300 x 32768 x 4096 596 / 587.  (The matrix whose rows a wave fetches is the same for all of its lanes: as an offset a lane it cost a
// register, which went to scratch memory in the loop, 2,840 beside 2,877 apart.)
template <int BM, int BN, int WM, int WN, bool CUT, bool GLU>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64)
gemm_f32_tile_kernel(float* __restrict__ C, const float* __restrict__ X, const float* __restrict__ W,
                     const float* __restrict__ bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha,
                     int m_tiles, int n_tiles, int vec_store, float* __restrict__ ws, const FtCut cut, int act) {
    constexpr int NW = (BM / WM) * (BN / WN), NT = NW * 64, ROWS = BM + BN;
    constexpr int LOADS = ROWS * 8 / NT, W_LOADS = BN * 8 / NT, TM = WM / 16, TN = WN / 16;
    static_assert(ROWS * 8 % NT == 0 && BN * 8 % NT == 0, "whole loads");
    // [stage][group of 16 rows (of W, then of X)][piece][slot]
    __shared__ __align__(16) uint4 lds[2][ROWS / 16][3][64];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int wn = (wave % (BN / WN)) * TN, wm = BN / 16 + (wave / (BN / WN)) * TM;   // the wave's first row groups
    const bool early = wave < NW / 2;

    const int stages = (K + F3_STEP - 1) / F3_STEP;
    const int per = (stages + F3_SLICES - 1) / F3_SLICES;
    const int k4_last = (K >> 2) - 1;

    // a thread stages 16 bytes (piece tid % 8 of a row's 128) of LOADS rows: tid / 8 + i * NT / 8
    const int lrow = tid >> 3, lk4 = tid & 7;
    // (in 16 bytes: a row of the tile, the tile's last row inside the matrix; rows beyond are that one again)
    const uint32_t w4 = ldw >> 2, x4 = lda >> 2;
    // (GLU: a wave's rows are all of gate or all of up; NT / 8 rows of the tile on are NT / 16 rows on of the same)
    const int up = GLU ? wave >> 1 & 1 : 0;
    const uint32_t w_each = (GLU ? NT / 16 : NT / 8) * w4;
    uint32_t wfrom = (GLU ? (lrow >> 5) * 16 + (lrow & 15) : lrow) * w4, xfrom = lrow * x4;
    const int put = (lrow >> 4) * 384 + f3_slot(lrow & 15, lk4 & 3) * 2 + (lk4 >> 2);   // in 8 bytes
    const int get = f3_slot(r, q);
    float4 reg[LOADS];
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    f32x4 acc[TN][TM], total[CUT ? 1 : TN][CUT ? 1 : TM];
    const int tile = CUT ? cut.first + (int)blockIdx.x / cut.parts : blockIdx.x, part = CUT ? blockIdx.x % cut.parts : 0;
    const int slice0 = CUT ? part * cut.slices / cut.parts : 0;
    const int st0 = slice0 * per, st1 = CUT ? min((part + 1) * cut.slices / cut.parts * per, stages) : stages;
    int mt, nt;
    ft_place(tile, m_tiles, n_tiles, mt, nt);
    const int n0 = nt * (GLU ? BN / 2 : BN), m0 = mt * BM;
    const float4* wsrc = reinterpret_cast<const float4*>(W + (size_t)(n0 + up * N) * ldw);
    const float4* xsrc = reinterpret_cast<const float4*>(X + (size_t)m0 * lda);
    const uint32_t wlast = (uint32_t)min(N - 1 - n0, (GLU ? BN / 2 : BN) - 1) * w4, xlast = (uint32_t)min(M - 1 - m0, BM - 1) * x4;
    auto fetch = [&](int st) {
        const int k4 = st * 8 + lk4, k4c = k4 < k4_last ? k4 : k4_last;
        asm volatile("" : "+v"(wfrom), "+v"(xfrom));   // the rows' offsets are made here each time: outside the loop they would take LOADS registers
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) reg[i] = wsrc[min(wfrom + i * w_each, wlast) + (uint32_t)k4c];
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

    // a slice's sums, as the waves hold them: [cut tile][slice][wave][t][g][lane]
    auto leave = [&](int slice) {
        f32x4* to = reinterpret_cast<f32x4*>(ws) + (((size_t)(tile - cut.first) * cut.slices + slice) * NW + wave) * (TN * TM * 64) + lane;
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int g = 0; g < TM; ++g) to[(t * TM + g) * 64] = acc[t][g];
    };
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int g = 0; g < TM; ++g) {
            acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (!CUT) total[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    fetch(st0);
    store(st0);
    fetch(st0 + 1);
    __syncthreads();
    int in_slice = 0, slice = slice0;
    for (int st = st0; st < st1; ++st) {
        if (early && st + 1 < st1) {
            store(st + 1);
            fetch(st + 2);
        }
        if (in_slice == per) {   // a slice ends: its sum joins the total, the next starts from zero
            in_slice = 0;
            if (CUT) leave(slice++);
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int g = 0; g < TM; ++g) {
                    if (!CUT) total[t][g] += acc[t][g];
                    acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        ++in_slice;
        // two tiles of W at a time: all of a wave's W fragments would take the registers that its sums need (LDS has room
        // for the second reading of X)
        __builtin_amdgcn_s_setprio(1);
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
        __builtin_amdgcn_s_setprio(0);
        if (!early && st + 1 < st1) {
            store(st + 1);
            fetch(st + 2);
        }
        __syncthreads();
    }
    if (CUT) {
        leave(slice);
        return;
    }
    unsigned long long open = 0;   // outputs to be computed again: bit (g * TN + t) * 4 + e
    static_assert(TM * TN * 4 <= 64, "a bit an output");
    if constexpr (GLU) {
        // acc[2 p][g][e] and acc[2 p + 1][g][e] of lane (r, q): gate and up of row m0 + 16 (wm's group + g) + r, output n0 + 16 (wn / 2 + p) + 4 q + e.
        // Where one of the two is to be computed again the other waits in its place in C; where both are, their product as it is (a NaN stays)
        auto biased = [&](float v, int n) { return bias != nullptr ? v + bias[n] : v; };
#pragma unroll
        for (int g = 0; g < TM; ++g) {
            const int m = m0 + (wm - BN / 16 + g) * 16 + r;
            if (m >= M) continue;
#pragma unroll
            for (int t = 0; t < TN; t += 2) {
                const int n = n0 + (wn + t) * 8 + 4 * q;
                if (n >= N) continue;
                const f32x4 vg = total[t][g] + acc[t][g], vu = total[t + 1][g] + acc[t + 1][g];
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (n + e >= N) continue;
                    const bool og = f3_unsaid(vg[e]), ou = f3_unsaid(vu[e]);
                    if (og) open |= 1ull << ((g * TN + t) * 4 + e);
                    if (ou) open |= 1ull << ((g * TN + t + 1) * 4 + e);
                    const float gate = biased(vg[e], n + e), u = biased(vu[e], N + n + e);
                    o[e] = og && !ou ? u : (ou && !og ? gate : glu_act(gate, act) * u);
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
        for (unsigned long long lanes; (lanes = __builtin_amdgcn_ballot_w64(open != 0ull)) != 0ull;) {
            const int owner = __builtin_ctzll(lanes);
            const bool mine = lane == owner;
            const int bit = __builtin_amdgcn_readlane(open != 0ull ? __builtin_ctzll(open) : 0, owner), g = bit / (4 * TN);
            const int first = bit - ((bit >> 2) & 1) * 4;   // the gate's bit; up's is four on
            const int which = __builtin_amdgcn_readlane((int)(open >> first & 0x11ull), owner);
            const int m = m0 + (wm - BN / 16 + g) * 16 + (owner & 15);
            const int n = n0 + (wn + first / 4 % TN) * 8 + 4 * (owner >> 4) + (first & 3);
            const float* x = X + (size_t)m * lda;
            if (f3_has_nan(x, K)) {   // (NaNs are there already, all along the row)
                if (mine) open &= ~(((1ull << (4 * TN)) - 1) << (4 * TN * g));
                continue;
            }
            float gate = 0.f, u = 0.f;
            if (which & 1) gate = biased(f3_dot(x, W + (size_t)n * ldw, K), n);
            if (which & 16) u = biased(f3_dot(x, W + (size_t)(N + n) * ldw, K), N + n);
            if (mine) {
                float* dst = C + (size_t)m * ldc + n;
                if (which == 1) u = *dst;
                if (which == 16) gate = *dst;
                *dst = glu_act(gate, act) * u;
                open &= ~(0x11ull << first);
            }
        }
        return;
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
            f32x4 v = total[CUT ? 0 : t][CUT ? 0 : g] + acc[t][g];
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = v[e];
                if (n + e < N && f3_unsaid(x)) open |= 1ull << ((g * TN + t) * 4 + e);
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
    // (as f3_settle, lane by lane)
    for (unsigned long long lanes; (lanes = __builtin_amdgcn_ballot_w64(open != 0ull)) != 0ull;) {
        const int owner = __builtin_ctzll(lanes);
        const bool mine = lane == owner;
        const int bit = __builtin_amdgcn_readlane(open != 0ull ? __builtin_ctzll(open) : 0, owner), g = bit / (4 * TN);
        const int m = m0 + (wm - BN / 16 + g) * 16 + (owner & 15);
        const int n = n0 + (wn + bit / 4 % TN) * 16 + 4 * (owner >> 4) + (bit & 3);
        const float* x = X + (size_t)m * lda;
        if (f3_has_nan(x, K)) {   // (NaNs are there already, all along the row)
            if (mine) open &= ~(((1ull << (4 * TN)) - 1) << (4 * TN * g));
            continue;
        }
        float v = f3_dot(x, W + (size_t)n * ldw, K);
        if (bias != nullptr) v += bias[n];
        if (mine) {
            C[(size_t)m * ldc + n] = alpha * v;
            open &= open - 1;
        }
    }
}

// Cut tiles: the slices' sums in ascending order.  A thread takes the four outputs that a lane of the tile's workgroup held together (GLU: those
// of gate and of up).
template <int BM, int BN, int WM, int WN, bool GLU>
__global__ void __launch_bounds__(256)
gemm_f32_sum_kernel(float* __restrict__ C, const float* __restrict__ ws, const float* __restrict__ X, const float* __restrict__ W,
                    const float* __restrict__ bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int m_tiles, int n_tiles,
                    int vec_store, const FtCut cut, int act) {
    constexpr int TM = WM / 16, TN = WN / 16, OF = GLU ? 2 : 1, EACH = BM * BN / 4, THREADS = EACH / OF;   // threads a tile
    const int tile = cut.first + blockIdx.x / (THREADS / 256);
    const int i = blockIdx.x % (THREADS / 256) * 256 + threadIdx.x, lane = i & 63, r = lane & 15, q = lane >> 4;
    const int g = i / 64 % TM, t = i / (64 * TM) % (TN / OF), wave = i / (64 * TM * (TN / OF));
    const f32x4* from = reinterpret_cast<const f32x4*>(ws) + (size_t)(tile - cut.first) * cut.slices * EACH + ((wave * TN + t * OF) * TM + g) * 64 + lane;
    f32x4 s[OF][F3_SLICES], v[OF];
#pragma unroll
    for (int h = 0; h < OF; ++h)
#pragma unroll
        for (int k = 0; k < F3_SLICES; ++k) s[h][k] = from[(size_t)(k < cut.slices ? k : 0) * EACH + h * TM * 64];
#pragma unroll
    for (int h = 0; h < OF; ++h) {
        v[h] = s[h][0];
#pragma unroll
        for (int k = 1; k < F3_SLICES; ++k)
            if (k < cut.slices) v[h] += s[h][k];
    }
    int mt, nt;
    ft_place(tile, m_tiles, n_tiles, mt, nt);
    const int m = mt * BM + (wave / (BN / WN) * TM + g) * 16 + r, n = nt * (BN / OF) + (wave % (BN / WN) * (TN / OF) + t) * 16 + 4 * q;
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const bool live = m < M && n + e < N;
        float x = f3_settle(v[0][e], live, X, W, m, n + e, K, lda, ldw);
        if (bias != nullptr && live) x += bias[n + e];
        if (GLU) {
            float u = f3_settle(v[OF - 1][e], live, X, W, m, N + n + e, K, lda, ldw);
            if (bias != nullptr && live) u += bias[N + n + e];
            o[e] = glu_act(x, act) * u;
        } else {
            o[e] = alpha * x;
        }
    }
    if (m >= M || n >= N) return;
    float* dst = C + (size_t)m * ldc + n;
    if (vec_store && n + 3 < N) {
        *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = o[e];
    }
}

// Which of the three tiles, or 4: the first, with the tiles beyond whole rounds cut (`parts` workgroups a tile)
static int ft_form(int M, int N, int K, int slices, int* parts) {
    // What ends soonest, by what a round of each takes (us at K 4096, measured on 256 units: the ratios count).  128 x
    // 256 and 128 x 128 run one a unit, 325 and 197 a round; of 64 x 64 three share a unit: 95 alone, 142 two of them, 190 three
    // (1024 x 2112 to 1024 x 3072: 184 to 197), 265 four, 66 each when many follow one another.  2048 x 4096 outputs: 368, 405 and 529 us; 300 x 4608: 324, 197 and 142.
    const long long cus = ilm_num_cus();
    auto count = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    const long long n1 = count(128, 256), t1 = 325 * ((n1 + cus - 1) / cus), t2 = 197 * ((count(128, 128) + cus - 1) / cus);
    const long long n3 = count(64, 64), t3 = n3 <= cus ? 95 : n3 <= 2 * cus ? 142 : n3 <= 3 * cus ? 190 : n3 <= 4 * cus ? 265 : 66 * n3 / cus + 10;
    const int form = t1 <= t2 && t1 <= t3 ? 1 : t2 <= t3 ? 2 : 3;
    const long long rest = n1 % cus;
    if (rest == 0 || slices < 2) return form;
    // Cut: rounds of workgroups of some slices each and 3 us for the start of a round, then the sum, 4 us and 0.03 a slice of a tile (128 KB, written and
    // read).  By this rule / measured, and the best whole form: 2048 x 4608 x 4096 380 / 382 (544), 1024 x 4608 x 4096 257 / 233 (305), 300 x 4608
    // x 4096 101 / 93 (138), 100 x 4608 x 4096 52 / 51 (97), 1024 x 4096 x 4096 200 / 188 (197), 2048 x 2304 x 2304 168 / 152 (178),
    // 1024 x 2304 x 2304 93 / 85 (106), 2048 x 1024 x 1024 43 / 44 (40), 2048 x 1280 x 1024 57 / 54 (52), 1024 x 6912 x 2304 237 / 228 (186), 1300 x 2048 x
    // 12288 400 / 362 (532).
    const double unit = 325. / 4096 * K / slices;
    double best = 0.;
    for (int p = 2; p <= slices; ++p) {
        const double t = (double)((rest * p + cus - 1) / cus) * (unit * ((slices + p - 1) / p) + 3.);
        if (p == 2 || t < best) best = t, *parts = p;
    }
    best += n1 / cus * 325. / 4096 * K + 4. + 0.03 * (double)(rest * slices);
    return best < (form == 1 ? t1 : form == 2 ? t2 : t3) / 4096. * K ? 4 : form;
}
static int ft_slices(int K) {
    const int steps = (K + F3_STEP - 1) / F3_STEP, per = (steps + F3_SLICES - 1) / F3_SLICES;
    return (steps + per - 1) / per;
}
static int ft_rest(int M, int N) { return (int)((long long)((M + 127) / 128) * ((N + 255) / 256) % ilm_num_cus()); }

static int ft_check(const char* name, const void* X, const void* W, int M, int N, int K, int lda, int ldw, int ldc) {
    ILM_REQUIRE(M > 0 && N > 0 && K > 0, "%s: bad sizes M=%d N=%d K=%d", name, M, N, K);
    ILM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda >= K && ldw >= K && ldc >= N,
                "%s: K=%d lda=%d ldw=%d ldc=%d", name, K, lda, ldw, ldc);
    ILM_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "%s: operands must be 16-byte aligned", name);
    ILM_REQUIRE(lda < (1 << 24) && ldw < (1 << 24), "%s: rows of %d and %d floats", name, lda, ldw);   // (offsets inside a tile take 32 bits)
    ILM_REQUIRE((long long)((M + 63) / 64) * ((N + 63) / 64) < (1ll << 31), "%s: too many tiles", name);
    return 0;
}
#define FT_ARGS (float*)C, (const float*)X, (const float*)W, (const float*)bias, M, N, K, lda, ldw, ldc, alpha
#define FT_RUN(BM_, BN_, WM_, WN_, CUT_, GLU_, BLOCKS_)                                                                       \
    {                                                                                                                   \
        const int m_tiles = (M + BM_ - 1) / BM_, n_tiles = ((GLU_ ? 2 : 1) * N + BN_ - 1) / BN_;                         \
        gemm_f32_tile_kernel<BM_, BN_, WM_, WN_, CUT_, GLU_><<<BLOCKS_, (BM_ / WM_) * (BN_ / WN_) * 64, 0, stream>>>(   \
            FT_ARGS, m_tiles, n_tiles, vec_store, (float*)ws, cut, act);                                                \
        ILM_LAUNCH_CHECK("gemm_f32_tile");                                                                              \
    }

// `tile`: 0 the rule above, 1 .. 3 one of the three shapes (for measurements and tests)
extern "C" int ilm_gemm_f32_tile(void* C, const void* X, const void* W, const void* bias, int M, int N, int K,
                                 int lda, int ldw, int ldc, float alpha, int tile, hipStream_t stream) {
    if (ft_check("gemm_f32_tile", X, W, M, N, K, lda, ldw, ldc) != 0) return -1;
    ILM_REQUIRE(tile >= 0 && tile <= 3, "gemm_f32_tile: there is no tile %d", tile);
    const int vec_store = (ldc % 4 == 0 && ((uintptr_t)C & 15) == 0) ? 1 : 0;
    int parts;
    void* ws = nullptr;
    const FtCut cut = {};
    const int act = 0;
    if (tile == 0) tile = ft_form(M, N, K, 1, &parts);   // (of the whole forms)
    if (tile == 1) FT_RUN(128, 256, 64, 64, false, false, m_tiles * n_tiles)
    else if (tile == 2) FT_RUN(128, 128, 64, 32, false, false, m_tiles * n_tiles)
    else FT_RUN(64, 64, 32, 32, false, false, m_tiles * n_tiles)
    return 0;
}

// Floats of the workspace that the form with cut tiles takes, or 0 where one of the others ends sooner.  At most the units less one times eight slices of
// 128 KB, whatever the sizes: 267 MB on 256 units.
extern "C" long ilm_gemm_f32_cut_ws(int M, int N, int K) {
    int parts;
    if (M <= 0 || N <= 0 || K <= 0 || ft_form(M, N, K, ft_slices(K), &parts) != 4) return 0;
    return (long)ft_rest(M, N) * ft_slices(K) * 128 * 256;
}

template <bool GLU>
static int ft_cut(void* C, const void* X, const void* W, const void* bias, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int act,
                  int parts, void* ws, long ws_floats, hipStream_t stream) {
    const int rows = GLU ? 2 * N : N, slices = ft_slices(K), rest = ft_rest(M, rows), m_tiles = (M + 127) / 128, n_tiles = (rows + 255) / 256;
    int rule = slices;
    ft_form(M, rows, K, slices, &rule);
    if (parts == 0) parts = rule;
    ILM_REQUIRE(parts >= 1 && parts <= slices, "gemm_f32_cut: %d workgroups for %d slices", parts, slices);
    ILM_REQUIRE(rest > 0 && ws != nullptr && ((uintptr_t)ws & 15) == 0 && ws_floats >= (long)rest * slices * 128 * 256,
                "gemm_f32_cut: %d tiles of %d slices, a workspace of %ld floats", rest, slices, ws_floats);
    const int vec_store = (ldc % 4 == 0 && ((uintptr_t)C & 15) == 0) ? 1 : 0;
    const FtCut cut = {m_tiles * n_tiles - rest, slices, parts};
    if (cut.first > 0) FT_RUN(128, 256, 64, 64, false, GLU, cut.first)
    FT_RUN(128, 256, 64, 64, true, GLU, rest * parts)
    gemm_f32_sum_kernel<128, 256, 64, 64, GLU><<<rest * (128 * 256 / 1024) / (GLU ? 2 : 1), 256, 0, stream>>>(
        (float*)C, (const float*)ws, (const float*)X, (const float*)W, (const float*)bias, M, N, K, lda, ldw, ldc, alpha, m_tiles, n_tiles, vec_store,
        cut, act);
    ILM_LAUNCH_CHECK("gemm_f32_sum");
    return 0;
}

// The same product with the tiles beyond whole rounds cut into their slices of K.  ws: ws_floats floats, at least as many as slices of such tiles hold.
// `parts`: workgroups a tile, 0 the rule's.
extern "C" int ilm_gemm_f32_cut(void* C, const void* X, const void* W, const void* bias, int M, int N, int K, int lda, int ldw, int ldc,
                                float alpha, int parts, void* ws, long ws_floats, hipStream_t stream) {
    if (ft_check("gemm_f32_cut", X, W, M, N, K, lda, ldw, ldc) != 0) return -1;
    return ft_cut<false>(C, X, W, bias, M, N, K, lda, ldw, ldc, alpha, 0, parts, ws, ws_floats, stream);
}

// act(X Wg^T + bg) * (X Wu^T + bu), W = [Wg; Wu] with I rows each, in tiles of 128 rows and 128 outputs.  Whether these are the rule's for the product
// alone (the smaller ones keep the activation apart), and that product's workspace
extern "C" int ilm_gemm_f32_glu_tile_ok(int M, int I, int K) {
    int parts;
    if (M <= 0 || I <= 0 || K <= 0 || I >= 1 << 30) return 0;
    const int form = ft_form(M, 2 * I, K, ft_slices(K), &parts);
    return form == 1 || form == 4 ? 1 : 0;
}
// ws: null, or ilm_gemm_f32_cut_ws(M, 2 I, K) floats: with cut tiles
extern "C" int ilm_gemm_f32_glu_tile(void* C, const void* X, const void* W, const void* bias, int M, int I, int K, int lda, int ldw, int ldc, int act,
                                     void* ws, long ws_floats, hipStream_t stream) {
    if (ft_check("gemm_f32_glu_tile", X, W, M, I, K, lda, ldw, ldc) != 0) return -1;
    ILM_REQUIRE(I < 1 << 30, "gemm_f32_glu_tile: %d outputs", I);
    const int N = I;
    const float alpha = 1.f;
    if (ws != nullptr) return ft_cut<true>(C, X, W, bias, M, N, K, lda, ldw, ldc, alpha, act, 0, ws, ws_floats, stream);
    const int vec_store = (ldc % 4 == 0 && ((uintptr_t)C & 15) == 0) ? 1 : 0;
    const FtCut cut = {};
    FT_RUN(128, 256, 64, 64, false, true, m_tiles * n_tiles)
    return 0;
}
#undef FT_RUN
#undef FT_ARGS
