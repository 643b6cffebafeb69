// Sampling from rows of float logits: argmax, and temperature / top-k / top-p with an inverse CDF.
//
// Definition: temperature == 0 or top_k == 1 -> the first index of the maximum.  Otherwise
// e_i = exp((l_i - max) / temperature); keep the top_k largest logits (0 or >= V keeps all; ties
// with the k-th value are kept); among those keep the fewest largest whose mass reaches top_p of
// the kept mass (ties kept); the token is the first index, in vocabulary order over the kept set,
// whose running mass exceeds u * (kept mass), u in [0, 1) supplied by the host per row.
//
// The thresholds come from histograms and not from a search bit by bit: the logits' distance from the maximum
// falls into 2,048 equal bins of 1/64 temperature, the bin that holds the threshold is found by one scan, its
// elements (a few hundred at most in a bin so narrow) are collected and ranked against each other.  Only a bin
// with more than LIST_CAP elements (rows of ties, everything beyond 32 temperatures) is searched by
// radix over the keys, three more passes.  Under a top-k of up to some thousand all that is kept fits the list, and
// the rest of the work happens there.
//
// What bounds it is arithmetic, some 40 instructions an element and pass for its mass and bin: one compute unit a row takes
// 110 us for 122,753 elements.  So few long rows are cut into chunks over the chip, four short kernels
// one after the other (maximum; histogram; list and masses of 256-element tiles; the token), the rows' results meeting in
// a workspace, and only rows whose threshold falls where lists overflow are done again by one workgroup.
// A call with its host's work, against 32 + 32 rounds of bitwise search over a row in registers (or in memory beyond
// 98,304): 64 rows x 73,448 with top-k 50 and top-p 0.9 55 us against 187, 5 rows x 122,753 with top-p 0.95 58 against 802.
//
// Masses are summed as whole numbers (e * 2^43): every sum is exact in its terms whatever the order, so the
// result depends on no order of atomics, and finer than sums of floats.
#include "common.h"

#define SB 1024
#define SNW (SB / 64)
#define NBINS 2048
#define LIST_CAP 2048
#define MAX_TILES 4096
#define CHUNK_THREADS 512
#define MAX_CHUNKS 32

typedef unsigned long long u64;

__device__ __forceinline__ uint32_t okey(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_to_float(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

__device__ __forceinline__ void better(float& bv, int& bi, float v, int i) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

// f(index, value) for every element of the row, by all threads of the block: 16-byte loads from the first aligned
// element on (rows of an odd vocabulary begin anywhere), four of them in flight a thread.
template <int NT, class F>
__device__ __forceinline__ void over_row(const float* __restrict__ row, int V, F f) {
    const int lead = (int)((4 - (((uintptr_t)row >> 2) & 3)) & 3);
    const int head = lead < V ? lead : V;
    const int n4 = (V - head) >> 2, tail = head + 4 * n4;
    if ((int)threadIdx.x < head) f((int)threadIdx.x, row[threadIdx.x]);
    const float4* row4 = reinterpret_cast<const float4*>(row + head);
    for (int i = threadIdx.x; i < n4; i += 4 * NT) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = i + u * NT;
            v[u] = row4[j < n4 ? j : n4 - 1];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = i + u * NT;
            if (j < n4) {
                f(head + 4 * j, v[u].x);
                f(head + 4 * j + 1, v[u].y);
                f(head + 4 * j + 2, v[u].z);
                f(head + 4 * j + 3, v[u].w);
            }
        }
    }
    if (tail + (int)threadIdx.x < V) f(tail + (int)threadIdx.x, row[tail + threadIdx.x]);
}

// argmax of one row by the whole block (first index on ties; 0x7fffffff for a row of NaN); result valid in every thread
template <int NT>
__device__ int block_argmax(const float* __restrict__ row, int V, float* sv, int* si, float* out_max) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    over_row<NT>(row, V, [&](int i, float v) { better(bv, bi, v, i); });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float ov = __shfl_xor(bv, o, 64);
        int oi = __shfl_xor(bi, o, 64);
        better(bv, bi, ov, oi);
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
        sv[w] = bv;
        si[w] = bi;
    }
    __syncthreads();
    bv = sv[0];
    bi = si[0];
    for (int i = 1; i < NT / 64; ++i) better(bv, bi, sv[i], si[i]);
    *out_max = bv;
    return bi;
}

__global__ void __launch_bounds__(SB)
argmax_kernel(int* __restrict__ out, const float* __restrict__ logits, int V, int stride) {
    __shared__ float sv[SNW];
    __shared__ int si[SNW];
    float mx;
    const int bi = block_argmax<SB>(logits + (size_t)blockIdx.x * stride, V, sv, si, &mx);
    if (threadIdx.x == 0) out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
}

extern "C" int ilm_argmax(void* out, const void* logits, int n, int V, int stride,
                          hipStream_t stream) {
    ILM_REQUIRE(n > 0 && V > 0 && stride >= V, "argmax: bad sizes n=%d V=%d stride=%d", n, V, stride);
    argmax_kernel<<<n, SB, 0, stream>>>((int*)out, (const float*)logits, V, stride);
    ILM_LAUNCH_CHECK("argmax");
    return 0;
}

// ---- reductions over the block; every thread gets the result ----------------------------------------------
template <int NT, class T, class Op>
__device__ __forceinline__ T block_reduce(T v, T* red, Op op) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    T t = red[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) t = op(t, red[i]);
    return t;
}
template <int NT>
__device__ __forceinline__ u64 block_sum_u64(u64 v, u64* red) {
    return block_reduce<NT>(v, red, [](u64 a, u64 b) { return a + b; });
}
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* red) {
    return block_reduce<SB>(v, red, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// exp((l - max) / temperature) as a whole number of 2^-43 (fewer for vocabularies beyond a million: `cut`).  The exponent's
// rounding error is carried along (x log2(e) in two pieces), so the result is good to a float's last bits.
// NaN counts as no mass.  (No product meets a sum outside fmaf: every pass computes the same bits for an element.)
struct Mass {
    float mx, inv_t;
    int cut;
    __device__ __forceinline__ u64 operator()(float l) const {
        const float x = (l - mx) * inv_t;
        const float hi = x * 1.44269502162933349609375f;                       // log2(e) to 24 bits
        const float lo = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502162933349609375f, -hi));   // log2(e)'s further bits, and what hi lost
        const float e = __builtin_amdgcn_exp2f(hi);
        const float m = fmaf(e, lo * 0.693147181f, e) * 1048576.f;             // 2^20
        if (!(m > 0.f)) return 0;
        const uint32_t whole = (uint32_t)m;
        const uint32_t part = (uint32_t)((m - (float)whole) * 8388608.f);      // 2^23
        return (((u64)whole << 23) + part) >> cut;
    }
};

// The bin of a logit: its distance from the maximum in steps of 1/64 temperature.  It never falls as the logit
// falls, so all of a bin lies above all of the next.  The last bin takes the rest (and NaN).
__device__ __forceinline__ int bin_of(float l, float mx, float per) {
    const float x = (mx - l) * per;
    return x < (float)(NBINS - 1) ? (int)x : NBINS - 1;
}

// The first entry of hist (in order) at which base + the running sum reaches `need`; -1 if none does.  `before`: base + the
// sum of the entries ahead of it.
struct Found {
    int at;
    u64 before, in;
};
template <int NT>
__device__ Found find_in(const u64* hist, u64 base, double need, u64* red, Found* shared) {
    constexpr int PER = NBINS / NT;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    u64 mine[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        mine[i] = hist[threadIdx.x * PER + i];
        sum += mine[i];
    }
    u64 incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 n = __shfl_up(incl, o, 64);
        if (lane >= o) incl += n;
    }
    if (lane == 63) red[w] = incl;
    if (threadIdx.x == 0) shared->at = -1;
    __syncthreads();
    u64 run = base + incl - sum;
    for (int i = 0; i < w; ++i) run += red[i];
    if (!((double)run >= need)) {   // (not reached before this thread's entries)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!((double)run >= need) && (double)(run + mine[i]) >= need) {
                shared->at = threadIdx.x * PER + i;
                shared->before = run;
                shared->in = mine[i];
            }
            run += mine[i];
        }
    }
    __syncthreads();
    const Found f = *shared;
    __syncthreads();
    return f;
}

struct SampleLds {
    u64 hist[NBINS];
    u64 red[SNW];
    float sv[SNW];
    int si[SNW];
    Found found;
    int listed;
    int pick;
    struct {
        uint32_t key[LIST_CAP];
        int index[LIST_CAP];
        u64 mass[LIST_CAP];
    } list;
    u64 tile[MAX_TILES];
};

__device__ __forceinline__ void clear_hist(SampleLds& S) {
    __syncthreads();
    for (int i = threadIdx.x; i < NBINS; i += SB) S.hist[i] = 0;
    __syncthreads();
}

// Adds the elements that `take` lets through to the list; how many there were (beyond LIST_CAP none is stored).
template <class Take>
__device__ int collect(const float* row, int V, SampleLds& S, const Mass& mass, Take take) {
    __syncthreads();
    if (threadIdx.x == 0) S.listed = 0;
    __syncthreads();
    over_row<SB>(row, V, [&](int i, float l) {
        if (take(l)) {
            const int at = atomicAdd(&S.listed, 1);
            if (at < LIST_CAP) {
                S.list.key[at] = okey(l);
                S.list.index[at] = i;
                S.list.mass[at] = mass(l);
            }
        }
    });
    __syncthreads();
    return S.listed;
}

// S.hist[i] = the sum over the listed j of weigh(j, i), for every listed i: as many threads an element as there are, each
// with its part of the j (one element a thread walked a list of 200 in 12 us, an LDS latency a step)
template <class Weigh>
__device__ void weigh_list(SampleLds& S, int n, Weigh weigh) {
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += SB) S.hist[i] = 0;
    __syncthreads();
    int width = 64;
    while (width < n && width < SB) width *= 2;
    const int parts = SB / width, len = (n + parts - 1) / parts;
    const int j0 = (int)threadIdx.x / width * len, j1 = j0 + len < n ? j0 + len : n;
    for (int i = threadIdx.x & (width - 1); i < n; i += width) {
        u64 w = 0;
#pragma unroll 8
        for (int j = j0; j < j1; ++j) w += weigh(j, i);
        if (w != 0) atomicAdd(&S.hist[i], w);
    }
    __syncthreads();
}

// The largest key of the list at which base + the weight of the listed keys from it upwards reaches `need` (0: none).
// COUNT: every element weighs one; else its mass, and only keys from `least` on weigh anything.
template <bool COUNT>
__device__ uint32_t rank_list(SampleLds& S, int n, uint32_t least, u64 base, double need) {
    weigh_list(S, n, [&](int j, int i) { return S.list.key[j] >= S.list.key[i] ? (COUNT ? 1ull : S.list.mass[j]) : 0ull; });
    uint32_t best = 0;
    for (int i = threadIdx.x; i < n; i += SB) {
        const uint32_t key = S.list.key[i];
        if (key >= least && (double)(base + S.hist[i]) >= need && key > best) best = key;
    }
    return block_max_u32(best, (uint32_t*)S.red);
}

// The largest key at which base + the weight of the elements of bin `bin` with keys from it upwards reaches `need`, by
// radix over the keys' 32 bits: for bins that the list does not hold.
template <bool COUNT>
__device__ uint32_t radix_bin(const float* row, int V, SampleLds& S, const Mass& mass, int bin, float per, uint32_t least, u64 base,
                              double need) {
    uint32_t prefix = 0, mask = 0;
    for (int level = 0; level < 3; ++level) {
        const int shift = level == 0 ? 21 : level == 1 ? 10 : 0;
        const uint32_t digits = level == 2 ? 1024 : 2048;
        clear_hist(S);
        over_row<SB>(row, V, [&](int, float l) {
            const uint32_t key = okey(l);
            const bool in = key >= least && (key & mask) == prefix && bin_of(l, mass.mx, per) == bin;
            const int at = (int)(digits - 1 - ((key >> shift) & (digits - 1)));
            const u64 w = in ? (COUNT ? 1ull : mass(l)) : 0ull;
            // rows of ties send all lanes to one entry: those that agree with the first lane add once
            const bool same = in && at == __builtin_amdgcn_readfirstlane(at);
            u64 sum = same ? w : 0ull;
            if (COUNT) {
                const u64 votes = __builtin_amdgcn_ballot_w64(same);
                if (same && (int)(threadIdx.x & 63) == __builtin_ctzll(votes)) atomicAdd(&S.hist[at], (u64)__popcll(votes));
            } else if (same && sum != 0) {
                atomicAdd(&S.hist[at], sum);
            }
            if (in && !same && w != 0) atomicAdd(&S.hist[at], w);
        });
        const Found f = find_in<SB>(S.hist, base, need, S.red, &S.found);
        if (f.at < 0) return 0;
        base = f.before;
        prefix |= (digits - 1 - (uint32_t)f.at) << shift;
        mask |= (digits - 1) << shift;
    }
    return prefix;
}

// tau of a top-p over what the list holds from `tau` on
__device__ uint32_t top_p_of_list(SampleLds& S, int listed, uint32_t tau, float pp) {
    u64 total = 0;
    for (int i = threadIdx.x; i < listed; i += SB) total += S.list.key[i] >= tau ? S.list.mass[i] : 0ull;
    total = block_sum_u64<SB>(total, S.red);
    return total > 0 ? rank_list<false>(S, listed, tau, 0, (double)pp * (double)total) : 0;
}

// Inverse CDF in vocabulary order over the list's elements from `tau` on
__device__ void token_of_list(SampleLds& S, int listed, uint32_t tau, float uniform, int amax, int* out) {
    if (threadIdx.x == 0) S.pick = 0x7fffffff;
    u64 total = 0;
    for (int i = threadIdx.x; i < listed; i += SB) total += S.list.key[i] >= tau ? S.list.mass[i] : 0ull;
    total = block_sum_u64<SB>(total, S.red);
    const double target = (double)uniform * (double)total;
    weigh_list(S, listed, [&](int j, int i) { return S.list.key[j] >= tau && S.list.index[j] <= S.list.index[i] ? S.list.mass[j] : 0ull; });
    for (int i = threadIdx.x; i < listed; i += SB)
        if (S.list.key[i] >= tau && S.list.mass[i] > 0 && target < (double)S.hist[i]) atomicMin(&S.pick, S.list.index[i]);
    __syncthreads();
    if (S.pick == 0x7fffffff) {   // no mass at all (an infinite maximum): the last kept element
        __syncthreads();
        if (threadIdx.x == 0) S.pick = -1;
        __syncthreads();
        for (int i = threadIdx.x; i < listed; i += SB)
            if (S.list.key[i] >= tau) atomicMax(&S.pick, S.list.index[i]);
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = S.pick >= 0 ? S.pick : amax;
}

// Tiles of 256 m consecutive elements, m = 1 up to a vocabulary of a million
__device__ __forceinline__ int tile_groups(int V) { return (V + 256 * MAX_TILES - 1) / (256 * MAX_TILES); }

// f(index, value) for the four elements of every lane in tile t (a wave's work); 16-byte loads where the row is aligned
template <class F>
__device__ __forceinline__ void over_tile(const float* __restrict__ row, int V, int t, int m, F f) {
    const bool whole = ((uintptr_t)row & 15) == 0;
    for (int g = 0; g < m; ++g) {
        const int i0 = (t * m + g) * 256 + 4 * (int)(threadIdx.x & 63);
        float l[4];
        if (whole && i0 + 3 < V) {
            const float4 v = *reinterpret_cast<const float4*>(row + i0);
            l[0] = v.x, l[1] = v.y, l[2] = v.z, l[3] = v.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) l[e] = row[i0 + e < V ? i0 + e : V - 1];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i0 + e < V) f(i0 + e, l[e]);
    }
}

__device__ __forceinline__ u64 wave_sum_u64(u64 v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Inverse CDF in vocabulary order over the row's elements from `tau` on, S.tile holding their tiles' masses: the tile that
// holds u * total, and in it the element.  `last`: the last kept element, taken where there is no mass at all.  The first wave.
__device__ void token_of_tiles(SampleLds& S, const float* row, int V, const Mass& mass, uint32_t tau, float uniform, int last, int amax,
                               int* out) {
    const int lane = threadIdx.x & 63, m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    const int stretch = (tiles + 63) / 64;   // a contiguous stretch of tiles a lane
    u64 mine = 0;
    for (int i = 0; i < stretch; ++i) mine += lane * stretch + i < tiles ? S.tile[lane * stretch + i] : 0ull;
    u64 incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 n = __shfl_up(incl, o, 64);
        if (lane >= o) incl += n;
    }
    const u64 total = __shfl(incl, 63, 64);
    const double target = (double)uniform * (double)total;
    u64 votes = __builtin_amdgcn_ballot_w64(mine > 0 && target < (double)incl);
    if (votes == 0) {
        if (lane == 0) *out = last >= 0 ? last : amax;
        return;
    }
    const int owner = __builtin_ctzll(votes);
    u64 run = __shfl(incl - mine, owner, 64);
    int tile = owner * stretch;
    while (!(target < (double)(run + S.tile[tile]))) run += S.tile[tile++];   // (ends within the owner's stretch, whose sum passes the target)
    for (int g0 = 0; g0 < m; ++g0) {
        const int at = (tile * m + g0) * 256 + lane;
        float l[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) l[g] = row[at + 64 * g < V ? at + 64 * g : V - 1];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const u64 mine_e = at + 64 * g < V && okey(l[g]) >= tau ? mass(l[g]) : 0ull;
            u64 in = mine_e;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const u64 n = __shfl_up(in, o, 64);
                if (lane >= o) in += n;
            }
            votes = __builtin_amdgcn_ballot_w64(mine_e > 0 && target < (double)(run + in));
            if (votes != 0) {
                if (lane == 0) *out = at + 64 * g + __builtin_ctzll(votes);
                return;
            }
            run += __shfl(in, 63, 64);
        }
    }
    if (lane == 0) *out = last >= 0 ? last : amax;
}

// A whole row by one workgroup
__device__ void sample_row(SampleLds& S, const float* row, int V, float temp, int k, float pp, float uniform, int cut, int* out) {
    float mx;
    int amax = block_argmax<SB>(row, V, S.sv, S.si, &mx);
    if (amax == 0x7fffffff) amax = 0;
    if (temp == 0.0f || k == 1) {
        if (threadIdx.x == 0) *out = amax;
        return;
    }
    const Mass mass = {mx, 1.0f / temp, cut};
    const float per = 64.f * mass.inv_t;
    uint32_t tau = 0;   // what is kept: keys from tau on
    int listed = -1;    // >= 0: the list holds that many elements, all of the kept ones among them

    if (k > 0 && k < V) {
        // threshold of the top-k: the k-th largest key.  The last bin is not counted (under a mask most of a row falls there)
        clear_hist(S);
        over_row<SB>(row, V, [&](int, float l) {
            const int b = bin_of(l, mx, per);
            if (b < NBINS - 1) atomicAdd(&S.hist[b], 1ull);
        });
        const Found f = find_in<SB>(S.hist, 0, (double)k, S.red, &S.found);
        if (f.at >= 0 && f.before + f.in <= LIST_CAP) {
            listed = collect(row, V, S, mass, [&](float l) { return bin_of(l, mx, per) <= f.at; });
            tau = rank_list<true>(S, listed, 0, 0, (double)k);
        } else if (f.at >= 0) {
            tau = radix_bin<true>(row, V, S, mass, f.at, per, 0, f.before, (double)k);
        } else {
            u64 before = 0;
            for (int i = threadIdx.x; i < NBINS; i += SB) before += S.hist[i];
            before = block_sum_u64<SB>(before, S.red);
            tau = radix_bin<true>(row, V, S, mass, NBINS - 1, per, 0, before, (double)k);
        }
    }
    if (pp < 1.0f) {
        // threshold of the top-p within what is kept
        uint32_t tp = 0;
        if (listed >= 0) {
            tp = top_p_of_list(S, listed, tau, pp);
        } else {
            clear_hist(S);
            u64 rest = 0;
            over_row<SB>(row, V, [&](int, float l) {
                if (okey(l) >= tau) {
                    const u64 m = mass(l);
                    const int b = bin_of(l, mx, per);
                    if (b < NBINS - 1) atomicAdd(&S.hist[b], m);
                    else rest += m;
                }
            });
            __syncthreads();
            u64 before = 0;
            for (int i = threadIdx.x; i < NBINS; i += SB) before += S.hist[i];
            before = block_sum_u64<SB>(before, S.red);
            const u64 total = before + block_sum_u64<SB>(rest, S.red);
            const double need = (double)pp * (double)total;
            if (total > 0) {
                const Found f = find_in<SB>(S.hist, 0, need, S.red, &S.found);
                const int bin = f.at >= 0 ? f.at : NBINS - 1;
                const u64 base = f.at >= 0 ? f.before : before;
                const int n = collect(row, V, S, mass, [&](float l) { return okey(l) >= tau && bin_of(l, mx, per) == bin; });
                tp = n <= LIST_CAP ? rank_list<false>(S, n, tau, base, need) : radix_bin<false>(row, V, S, mass, bin, per, tau, base, need);
            }
        }
        if (!(pp > 0.f)) tp = okey(mx);
        if (tp > tau) tau = tp;
    }
    if (listed >= 0) {
        token_of_list(S, listed, tau, uniform, amax, out);
        return;
    }
    const int w = threadIdx.x >> 6, m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    int my_last = -1;
    for (int t = w; t < tiles; t += SNW) {
        u64 sum = 0;
        over_tile(row, V, t, m, [&](int i, float l) {
            if (okey(l) >= tau) {
                sum += mass(l);
                my_last = i;
            }
        });
        sum = wave_sum_u64(sum);
        if ((threadIdx.x & 63) == 0) S.tile[t] = sum;
    }
    const int last = (int)block_max_u32((uint32_t)(my_last + 1), (uint32_t*)S.red) - 1;
    if (w == 0) token_of_tiles(S, row, V, mass, tau, uniform, last, amax, out);
}

__global__ void __launch_bounds__(SB)
sample_kernel(int* __restrict__ out, const float* __restrict__ logits, const float* __restrict__ temperature,
              const int* __restrict__ top_k, const float* __restrict__ top_p,
              const float* __restrict__ uniform, int V, int stride, int cut) {
    __shared__ SampleLds S;
    const int r = blockIdx.x;
    sample_row(S, logits + (size_t)r * stride, V, temperature[r], top_k[r], top_p[r], uniform[r], cut, out + r);
}

// ---- rows in chunks ----------------------------------------------------------------------------------------
// What a row's chunks leave in the workspace.  The first kernel clears what later ones add to.
struct RowWork {
    u64 hist[NBINS];
    u64 rest;                   // mass of the last bin
    int listed, last;           // elements listed; the last element of the bins ahead of the threshold's, + 1
    float max_v[MAX_CHUNKS];
    int max_i[MAX_CHUNKS];
    uint32_t key[LIST_CAP];
    int index[LIST_CAP];
    u64 tile[1];                // (as many as the vocabulary has)
};

// The chunk's whole tiles [first, first + count)
struct Chunk {
    int first, count, begin, size;
};
__device__ __forceinline__ Chunk chunk_of(int V) {
    const int m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m), per = (tiles + (int)gridDim.x - 1) / (int)gridDim.x;
    Chunk c;
    c.first = blockIdx.x * per < tiles ? blockIdx.x * per : tiles;
    c.count = tiles - c.first < per ? tiles - c.first : per;
    c.begin = c.first * 256 * m;
    c.size = c.begin + c.count * 256 * m < V ? c.count * 256 * m : V - c.begin;
    if (c.size < 0) c.size = 0;
    return c;
}

__global__ void __launch_bounds__(CHUNK_THREADS)
sample_max_kernel(char* __restrict__ ws, size_t ws_row, const float* __restrict__ logits, int V, int stride) {
    __shared__ float sv[CHUNK_THREADS / 64];
    __shared__ int si[CHUNK_THREADS / 64];
    const int r = blockIdx.y;
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    for (int i = blockIdx.x * CHUNK_THREADS + threadIdx.x; i < NBINS; i += gridDim.x * CHUNK_THREADS) W->hist[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        W->rest = 0;
        W->listed = 0;
        W->last = 0;
    }
    const Chunk c = chunk_of(V);
    float mx = -INFINITY;
    int at = 0x7fffffff;
    if (c.size > 0) at = block_argmax<CHUNK_THREADS>(logits + (size_t)r * stride + c.begin, c.size, sv, si, &mx);
    if (threadIdx.x == 0) {
        W->max_v[blockIdx.x] = mx;
        W->max_i[blockIdx.x] = at == 0x7fffffff ? at : c.begin + at;
    }
}

__device__ __forceinline__ int row_max(const RowWork* W, int chunks, float* mx) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int i = 0; i < chunks; ++i) better(bv, bi, W->max_v[i], W->max_i[i]);
    *mx = bv;
    return bi == 0x7fffffff ? 0 : bi;
}

__global__ void __launch_bounds__(CHUNK_THREADS)
sample_hist_kernel(char* __restrict__ ws, size_t ws_row, const float* __restrict__ logits, const float* __restrict__ temperature,
                   const int* __restrict__ top_k, const float* __restrict__ top_p, int V, int stride, int cut) {
    __shared__ u64 hist[NBINS];
    __shared__ u64 red[CHUNK_THREADS / 64];
    const int r = blockIdx.y, k = top_k[r];
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float temp = temperature[r], pp = top_p[r];
    const bool count = k > 0 && k < V;
    if (temp == 0.0f || k == 1 || (!count && !(pp < 1.0f))) return;
    float mx;
    row_max(W, gridDim.x, &mx);
    const Mass mass = {mx, 1.0f / temp, cut};
    const float per = 64.f * mass.inv_t;
    for (int i = threadIdx.x; i < NBINS; i += CHUNK_THREADS) hist[i] = 0;
    __syncthreads();
    const Chunk c = chunk_of(V);
    u64 rest = 0;
    over_row<CHUNK_THREADS>(logits + (size_t)r * stride + c.begin, c.size, [&](int, float l) {
        const int b = bin_of(l, mx, per);
        const u64 w = count ? 1ull : mass(l);
        if (b < NBINS - 1) atomicAdd(&hist[b], w);
        else rest += w;
    });
    rest = block_sum_u64<CHUNK_THREADS>(rest, red);   // (its barriers close the histogram too)
    for (int i = threadIdx.x; i < NBINS; i += CHUNK_THREADS)
        if (hist[i] != 0) atomicAdd(&W->hist[i], hist[i]);
    if (threadIdx.x == 0 && rest != 0) atomicAdd(&W->rest, rest);
}

// Where the row's first threshold lies, from its histogram: found.at < 0 and no top-k or top-p: everything is kept; `whole`: the row
// is left to one workgroup (a threshold in the last bin, a top-k beyond the list, no mass, p not above 0)
template <int NT>
__device__ Found row_threshold(const RowWork* W, u64* red, Found* shared, bool count, int k, float pp, bool* whole, double* need) {
    Found f = {-1, 0, 0};
    *whole = false;
    *need = 0;
    if (!count && !(pp < 1.0f)) return f;
    if (count) {
        *need = (double)k;
    } else {
        u64 total = 0;
        for (int i = threadIdx.x; i < NBINS; i += NT) total += W->hist[i];
        total = block_sum_u64<NT>(total, red) + W->rest;
        *need = (double)pp * (double)total;
        if (!(pp > 0.f) || total == 0) {
            *whole = true;
            return f;
        }
    }
    f = find_in<NT>(W->hist, 0, *need, red, shared);
    *whole = f.at < 0 || (count && f.before + f.in > LIST_CAP);
    return f;
}

__global__ void __launch_bounds__(CHUNK_THREADS)
sample_list_kernel(char* __restrict__ ws, size_t ws_row, const float* __restrict__ logits, const float* __restrict__ temperature,
                   const int* __restrict__ top_k, const float* __restrict__ top_p, int V, int stride, int cut) {
    __shared__ u64 red[CHUNK_THREADS / 64];
    __shared__ Found shared;
    const int r = blockIdx.y, k = top_k[r];
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float* row = logits + (size_t)r * stride;
    const float temp = temperature[r], pp = top_p[r];
    const bool count = k > 0 && k < V;
    if (temp == 0.0f || k == 1) return;
    bool whole;
    double need;
    const Found f = row_threshold<CHUNK_THREADS>(W, red, &shared, count, k, pp, &whole, &need);
    if (whole) return;
    float mx;
    row_max(W, gridDim.x, &mx);
    const Mass mass = {mx, 1.0f / temp, cut};
    const float per = 64.f * mass.inv_t;
    auto list = [&](int i, float l) {
        const int at = atomicAdd(&W->listed, 1);
        if (at < LIST_CAP) {
            W->key[at] = okey(l);
            W->index[at] = i;
        }
    };
    const Chunk c = chunk_of(V);
    if (count) {   // everything down to the threshold's bin
        over_row<CHUNK_THREADS>(row + c.begin, c.size, [&](int i, float l) {
            if (bin_of(l, mx, per) <= f.at) list(c.begin + i, l);
        });
        return;
    }
    const int m = tile_groups(V), above = f.at >= 0 ? f.at : NBINS;   // the bins ahead of the threshold's are kept whole
    int my_last = -1;
    for (int t = c.first + (int)(threadIdx.x >> 6); t < c.first + c.count; t += CHUNK_THREADS / 64) {
        u64 sum = 0;
        over_tile(row, V, t, m, [&](int i, float l) {
            const int b = bin_of(l, mx, per);
            if (b < above) {
                sum += mass(l);
                my_last = i;
            } else if (b == above) {
                list(i, l);
            }
        });
        sum = wave_sum_u64(sum);
        if ((threadIdx.x & 63) == 0) W->tile[t] = sum;
    }
    if (my_last >= 0) atomicMax(&W->last, my_last + 1);
}

__global__ void __launch_bounds__(SB)
sample_token_kernel(int* __restrict__ out, char* __restrict__ ws, size_t ws_row, int chunks, const float* __restrict__ logits,
                    const float* __restrict__ temperature, const int* __restrict__ top_k, const float* __restrict__ top_p,
                    const float* __restrict__ uniform, int V, int stride, int cut) {
    __shared__ SampleLds S;
    const int r = blockIdx.x, k = top_k[r];
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float* row = logits + (size_t)r * stride;
    const float temp = temperature[r], pp = top_p[r];
    const bool count = k > 0 && k < V;
    float mx;
    const int amax = row_max(W, chunks, &mx);
    if (temp == 0.0f || k == 1) {
        if (threadIdx.x == 0) out[r] = amax;
        return;
    }
    bool whole;
    double need;
    const Found f = row_threshold<SB>(W, S.red, &S.found, count, k, pp, &whole, &need);
    const int listed = W->listed;
    if (whole || listed > LIST_CAP) {
        sample_row(S, row, V, temp, k, pp, uniform[r], cut, out + r);
        return;
    }
    const Mass mass = {mx, 1.0f / temp, cut};
    for (int i = threadIdx.x; i < listed; i += SB) {
        const uint32_t key = W->key[i];
        S.list.key[i] = key;
        S.list.index[i] = W->index[i];
        S.list.mass[i] = mass(key_to_float(key));
    }
    __syncthreads();
    if (count) {
        uint32_t tau = rank_list<true>(S, listed, 0, 0, need);
        if (pp < 1.0f) {
            const uint32_t tp = pp > 0.f ? top_p_of_list(S, listed, tau, pp) : okey(mx);
            if (tp > tau) tau = tp;
        }
        token_of_list(S, listed, tau, uniform[r], amax, out + r);
        return;
    }
    const uint32_t tau = f.at >= 0 ? rank_list<false>(S, listed, 0, f.before, need) : 0u;
    const int m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    for (int t = threadIdx.x; t < tiles; t += SB) S.tile[t] = W->tile[t];
    if (threadIdx.x == 0) S.pick = W->last;
    __syncthreads();
    for (int i = threadIdx.x; i < listed; i += SB)
        if (S.list.key[i] >= tau) {
            atomicAdd(&S.tile[S.list.index[i] / (256 * m)], S.list.mass[i]);
            atomicMax(&S.pick, S.list.index[i] + 1);
        }
    __syncthreads();
    if (threadIdx.x < 64) token_of_tiles(S, row, V, mass, tau, uniform[r], S.pick - 1, amax, out + r);
}

// Bytes of workspace a row needs of n rows of V logits; 0: none, the rows are not cut into chunks.  They are where few rows leave
// the chip idle and a row is long enough to outweigh three more launches.  In chunks against one workgroup a row, with top-p
// alone: 5 rows of 122,753 51 us against 110, 16 of 73,448 42 against 66, 64 of 32,768 43 against 38; with top-k 50, where
// less is computed, 1 row of 73,448 28 against 33, 64 of them 44 against 34.
extern "C" long ilm_sample_ws(int n, int V) {
    if (V <= 40960 || n > 32) return 0;
    return (long)(sizeof(RowWork) + sizeof(u64) * ((V + 255) / 256) + 15) / 16 * 16;
}

// `ws`: n * ilm_sample_ws(n, V) bytes, 16-byte aligned, or null: every row by one workgroup
extern "C" int ilm_sample(void* out, const void* logits, const void* temperature, const void* top_k,
                          const void* top_p, const void* uniform, void* ws, int n, int V, int stride,
                          hipStream_t stream) {
    ILM_REQUIRE(n > 0 && V > 0 && stride >= V, "sample: bad sizes n=%d V=%d stride=%d", n, V, stride);
    ILM_REQUIRE(((uintptr_t)ws & 15) == 0, "sample: the workspace must be 16-byte aligned");
    int cut = 0;   // V elements of at most 2^43 each: below 2^64 up to a vocabulary of 2^20
    while ((long long)V >> (20 + cut)) ++cut;
    const size_t ws_row = (size_t)ilm_sample_ws(n, V);
    if (ws == nullptr || ws_row == 0) {
        sample_kernel<<<n, SB, 0, stream>>>((int*)out, (const float*)logits, (const float*)temperature, (const int*)top_k,
                                            (const float*)top_p, (const float*)uniform, V, stride, cut);
        ILM_LAUNCH_CHECK("sample");
        return 0;
    }
    // chunks of at least 4,096 elements, up to four workgroups a compute unit
    int chunks = (V + 4095) / 4096;
    if (chunks > MAX_CHUNKS) chunks = MAX_CHUNKS;
    const int most = 4 * ilm_num_cus() / n;
    if (chunks > most) chunks = most;
    const dim3 grid(chunks, n);
    char* w = (char*)ws;
    sample_max_kernel<<<grid, CHUNK_THREADS, 0, stream>>>(w, ws_row, (const float*)logits, V, stride);
    sample_hist_kernel<<<grid, CHUNK_THREADS, 0, stream>>>(w, ws_row, (const float*)logits, (const float*)temperature, (const int*)top_k,
                                                           (const float*)top_p, V, stride, cut);
    sample_list_kernel<<<grid, CHUNK_THREADS, 0, stream>>>(w, ws_row, (const float*)logits, (const float*)temperature, (const int*)top_k,
                                                           (const float*)top_p, V, stride, cut);
    sample_token_kernel<<<n, SB, 0, stream>>>((int*)out, w, ws_row, chunks, (const float*)logits, (const float*)temperature,
                                              (const int*)top_k, (const float*)top_p, (const float*)uniform, V, stride, cut);
    ILM_LAUNCH_CHECK("sample");
    return 0;
}
