// Sampling from rows of float logits: argmax, and temperature / top-k / top-p with an inverse CDF.
//
// Definition: temperature == 0 or top_k == 1 -> the first index of the maximum.  Otherwise
// e_i = exp((l_i - max) / temperature); keep the top_k largest logits (0 or >= V keeps all; ties
// with the k-th value are kept); among those keep the fewest largest whose mass reaches top_p of
// the kept mass (ties kept); the token is the first index, in vocabulary order over the kept set,
// whose running mass exceeds u * (kept mass), u in [0, 1) supplied by the host per row.
//
// The thresholds come from histograms and not from a search bit by bit: the logits' distance from the maximum
// falls into 2,048 equal bins of 1/64 temperature (narrower ones for rows whose numbers lie close together), the bin that holds the threshold is found by one scan, its
// elements (a few hundred at most in a bin so narrow) are collected and ranked, against each other or, a long list, by radix in
// LDS.  Only a bin with more than LIST_CAP elements (rows of ties, everything beyond 32 temperatures) is searched by
// radix over the row's keys, three more passes, or one where all of the bin are the same number.  Under a top-k of up to
// some thousand all that is kept fits the list, and the rest of the work happens there.
//
// (What every row runs is inlined and what few do is called: left to the compiler, which function becomes a call
// changes with the code around it, at 1 to 30 us a call of the sampler.)
//
// What bounds it is arithmetic, some 40 instructions an element and pass for its mass and bin: one compute unit a row takes
// 103 us for 122,753 elements.  So few long rows are cut into chunks over the chip, four short kernels
// one after the other (maximum; histogram; list and masses of 256-element tiles; the token), the rows' results meeting in
// a workspace, and only rows whose threshold falls where lists overflow are done again by one workgroup.  A row with a small top-k
// needs neither masses nor bins for all of its elements (top_k_of_few).
// A call with its host's work, against histograms for every row (and 32 + 32 rounds of bitwise search before them): 64 rows x 73,448 with
// top-k 50 and top-p 0.9 33 us against 55 (187), 5 rows x 122,753 with top-p 0.95 37 against 49 (802), of which the kernels take 20 against 35
// and 30 (4.8, 6.4, 8.0 and 10.6) against 43 (4.9, 6.6, 14.1 and 17.5).
//
// Masses are summed as whole numbers (e * 2^43): every sum is exact in its terms whatever the order, so the
// result depends on no order of atomics, and finer than sums of floats.
#include "common.h"

#include <string.h>

#include <type_traits>

#define SB 1024
#define SNW (SB / 64)
#define NBINS 2048
#define LIST_CAP 2048
#define RANK_MAX 256    // listed elements up to which each is weighed against all others
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

// What a sample of a row tells, one number a lane, masked ones (-1e30 or less) left out: how many in a wave are the number
// of its first, less one, and that number (infinity where more than half are masked: a few may lie anywhere); of several waves the
// sum and the lowest
struct Sampled {
    int ties;
    float low;
};
__device__ __forceinline__ Sampled sample_of(float sample) {
    const u64 in = __builtin_amdgcn_ballot_w64(sample > -1e30f);
    if (in == 0ull) return {0, INFINITY};
    const float first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sample), __builtin_ctzll(in)));
    return {(int)__popcll(__builtin_amdgcn_ballot_w64(sample == first)) - 1, __popcll(in) < 32 ? INFINITY : first};
}

struct __align__(16) RowMax {
    float value;
    int index;      // 0x7fffffff: a row of NaN
    Sampled seen;
};

// argmax of one row by the whole block (first index on ties); result valid in every thread.  `seen`: a wave's sample; `meet`: a place a wave
template <int NT>
__device__ __forceinline__ RowMax block_argmax(const float* __restrict__ row, int V, Sampled seen, RowMax* meet) {
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
    if (lane == 0) meet[w] = {bv, bi, seen};
    __syncthreads();
    RowMax m = meet[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) {
        const RowMax o = meet[i];
        better(m.value, m.index, o.value, o.index);
        m.seen.ties += o.seen.ties;
        m.seen.low = fminf(m.seen.low, o.seen.low);
    }
    return m;
}

__global__ void __launch_bounds__(SB)
argmax_kernel(int* __restrict__ out, const float* __restrict__ logits, int V, int stride) {
    __shared__ RowMax meet[SNW];
    const RowMax m = block_argmax<SB>(logits + (size_t)blockIdx.x * stride, V, {0, 0.f}, meet);
    if (threadIdx.x == 0) out[blockIdx.x] = m.index == 0x7fffffff ? 0 : m.index;
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
// falls, so all of a bin lies above all of the next.  The last bin takes the rest (and NaN, which fminf drops).  The conversion saturates
// at zero: under a negative temperature the first bin holds all (a caller may hand one in: it lies on the device, where
// no one looks).  An instruction less than comparing before a conversion, two less with a clamp at zero.
__device__ __forceinline__ int bin_of(float l, float mx, float per) {
    const float x = fminf((mx - l) * per, (float)(NBINS - 1));
    uint32_t b;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(b) : "v"(x));
    return (int)b;
}

// Bins for a unit of a logit: 64 a temperature, or, where a row's numbers lie so close that they would share a few of those (its
// sample spans less than 128), so many that the sample spans half of them all.  The lanes of a wave that add to one bin wait for each
// other, and a bin of more than LIST_CAP elements takes three more passes: normal logits of a hundredth of the temperature, 64 rows of
// 73,448, top-k 50 104 us -> 32 (the search bit by bit 77), top-p 0.9 163 -> 66 (248); other rows pay 0.2 to 1 us.  Where the sample misleads,
// more falls into the last bin.
__device__ __forceinline__ float bins_per(float mx, float low, float inv_t) {
    const float per = 64.f * inv_t, spread = mx - low, bins = spread * per;
    return bins > 0.f && bins < 128.f ? (float)(NBINS / 2) / spread : per;
}

// The first entry of hist (in order) at which base + the running sum reaches `need`; -1 if none does.  `before`: base + the
// sum of the entries ahead of it.
struct Found {
    int at;
    u64 before, in;
};
template <int NT>
__device__ __forceinline__ Found find_in(const u64* hist, u64 base, double need, u64* red, Found* shared) {
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

// *to += w, by many lanes of a wave.  `like`: lanes with the same one add the same to the same place, and those that agree with
// the first lane add once.  LDS takes the lanes of one place one after the other, 0.8 ns each, so rows of ties would wait for that in every
// pass: 64 rows of 73,448 equal logits, top-p 0.95, 385 us instead of 89.
__device__ __forceinline__ void add_once(u64* to, u64 w, uint32_t like) {
    const bool first = like == __builtin_amdgcn_readfirstlane(like);
    const u64 same = __builtin_amdgcn_ballot_w64(first);
    const int count = __popcll(same);
    if (count > 1 && first) {
        if ((int)(threadIdx.x & 63) != __builtin_ctzll(same)) return;
        w *= (u64)count;
    }
    atomicAdd(to, w);
}

// Other rows lose 10 to 20 % by it, so the histograms of a row are made either way, as a sample of a number a thread tells: where TIE_SHARE
// of a wave's lanes or more agree with one of them (sample_of).  In bins as narrow as these one number in 450 meets another by
// chance (normal logits of deviation two at temperature 1).
#define TIE_SHARE 16    // (one in)

struct SampleLds {
    u64 hist[NBINS];
    u64 red[SNW];
    RowMax meet[SNW];
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
__device__ __forceinline__ int collect(const float* row, int V, SampleLds& S, const Mass& mass, Take take) {
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
__device__ __forceinline__ void weigh_list(SampleLds& S, int n, Weigh weigh) {
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

// The largest key at which base + the weight of the elements with keys from it upwards reaches `need` (0: none), by radix over the keys'
// 32 bits.  each(f) hands every element to f(key, weight of it), three times, or once if all have one key.  COUNT: an element weighs one.
template <bool COUNT, class Each>
__device__ __forceinline__ uint32_t radix_keys(SampleLds& S, u64 base, double need, Each each) {
    uint32_t prefix = 0, mask = 0, least = 0xffffffffu, most = 0;
    for (int level = 0; level < 3; ++level) {
        const int shift = level == 0 ? 21 : level == 1 ? 10 : 0;
        const uint32_t digits = level == 2 ? 1024 : 2048;
        clear_hist(S);
        each([&](uint32_t key, auto weight) {
            if ((key & mask) != prefix) return;
            least = key < least ? key : least;
            most = key > most ? key : most;
            const int at = (int)(digits - 1 - ((key >> shift) & (digits - 1)));
            add_once(&S.hist[at], COUNT ? 1ull : weight(), COUNT ? (uint32_t)at : key);
        });
        const Found f = find_in<SB>(S.hist, base, need, S.red, &S.found);
        if (f.at < 0) return 0;
        if (level == 0) {
            least = ~block_max_u32(~least, (uint32_t*)S.red);
            if (least == block_max_u32(most, (uint32_t*)S.red)) return least;
        }
        base = f.before;
        prefix |= (digits - 1 - (uint32_t)f.at) << shift;
        mask |= (digits - 1) << shift;
    }
    return prefix;
}

// ... of the elements of bin `bin` with keys from `least` on: for bins that the list does not hold
template <bool COUNT>
__device__ __noinline__ uint32_t radix_bin(const float* row, int V, SampleLds& S, Mass mass, int bin, float per, uint32_t least, u64 base,
                              double need) {
    return radix_keys<COUNT>(S, base, need, [&](auto f) {
        over_row<SB>(row, V, [&](int, float l) {
            const uint32_t key = okey(l);
            // (a NaN lies in the last bin with a key above all others': it counts towards nothing)
            if (key >= least && l == l && bin_of(l, mass.mx, per) == bin) f(key, [&]() { return mass(l); });
        });
    });
}

// ... of the list's elements with keys from `least` on: every one against all others, or by radix from where that takes longer
// (a row of 4,096, top-k and top-p: 200 listed 27 us; 1,000 194 with all against all and 27 by radix, 2,048 706 and 29)
template <bool COUNT>
__device__ __noinline__ uint32_t radix_list(SampleLds& S, int n, uint32_t least, u64 base, double need) {
    return radix_keys<COUNT>(S, base, need, [&](auto f) {
        for (int i = threadIdx.x; i < n; i += SB)
            if (S.list.key[i] >= least) f(S.list.key[i], [&]() { return S.list.mass[i]; });
    });
}
template <bool COUNT>
__device__ __forceinline__ uint32_t rank_list(SampleLds& S, int n, uint32_t least, u64 base, double need) {
    if (n > RANK_MAX) return radix_list<COUNT>(S, n, least, base, need);   // (a call: inlined, it slows the short lists by 1.5 us)
    weigh_list(S, n, [&](int j, int i) { return S.list.key[j] >= S.list.key[i] ? (COUNT ? 1ull : S.list.mass[j]) : 0ull; });
    uint32_t best = 0;
    for (int i = threadIdx.x; i < n; i += SB) {
        const uint32_t key = S.list.key[i];
        if (key >= least && (double)(base + S.hist[i]) >= need && key > best) best = key;
    }
    return block_max_u32(best, (uint32_t*)S.red);
}

// rank_list of one bin's elements, which lie even over a short range of keys: a long list falls into 2,048 steps of that range, one or two
// elements a step, and the step that holds the threshold is ranked by every wave for itself (one histogram instead of radix's three:
// 5 rows of 122,753, top-p 0.95, about 390 listed: the kernel that ends in it
// 14.3 -> 10.6 us).  Rows by one workgroup keep radix: inlined there too, this code cost short lists 0.3 us and gave long ones nothing
#define STEP_MAX 64
__device__ __forceinline__ uint32_t rank_bin(SampleLds& S, int n, uint32_t least, u64 base, double need) {
    if (n <= RANK_MAX) return rank_list<false>(S, n, least, base, need);
    u64 ends = 0;     // the largest key, and the largest complement of one
    for (int i = threadIdx.x; i < n; i += SB) {
        const uint32_t key = S.list.key[i];
        const u64 one = (u64)key << 32 | (uint32_t)~key;
        ends = i == (int)threadIdx.x ? one : ((ends >> 32) > key ? ends >> 32 : key) << 32 | ((uint32_t)ends > (uint32_t)~key ? (uint32_t)ends : (uint32_t)~key);
    }
    ends = block_reduce<SB>(ends, S.red, [](u64 a, u64 b) {
        const u64 h = (a >> 32) > (b >> 32) ? a >> 32 : b >> 32;
        return h << 32 | ((uint32_t)a > (uint32_t)b ? (uint32_t)a : (uint32_t)b);
    });
    const uint32_t hi = (uint32_t)(ends >> 32), range = hi - ~(uint32_t)ends;
    const int bits = range == 0 ? 0 : 32 - __builtin_clz(range), shift = bits > 11 ? bits - 11 : 0;
    clear_hist(S);
    for (int i = threadIdx.x; i < n; i += SB)
        if (S.list.key[i] >= least) atomicAdd(&S.hist[(hi - S.list.key[i]) >> shift], S.list.mass[i]);
    const Found f = find_in<SB>(S.hist, base, need, S.red, &S.found);
    if (f.at < 0) return 0;
    if (threadIdx.x == 0) S.listed = 0;
    __syncthreads();
    u64* mass = S.hist;                                              // of the step's elements, and behind them their keys
    uint32_t* key = reinterpret_cast<uint32_t*>(S.hist + STEP_MAX);
    for (int i = threadIdx.x; i < n; i += SB)
        if (S.list.key[i] >= least && (int)((hi - S.list.key[i]) >> shift) == f.at) {
            const int to = atomicAdd(&S.listed, 1);
            if (to < STEP_MAX) {
                mass[to] = S.list.mass[i];
                key[to] = S.list.key[i];
            }
        }
    __syncthreads();
    const int m = S.listed;
    if (m > STEP_MAX) return radix_list<false>(S, n, least, base, need);
    const int lane = threadIdx.x & 63;
    const uint32_t mine = lane < m ? key[lane] : 0u;
    u64 sum = f.before;
    for (int j = 0; j < m; ++j) sum += key[j] >= mine ? mass[j] : 0ull;
    uint32_t best = lane < m && (double)sum >= need ? mine : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t v = __shfl_xor(best, o, 64);
        best = v > best ? v : best;
    }
    return best;
}

// tau of a top-p over what the list holds from `tau` on
__device__ __forceinline__ uint32_t top_p_of_list(SampleLds& S, int listed, uint32_t tau, float pp) {
    u64 total = 0;
    for (int i = threadIdx.x; i < listed; i += SB) total += S.list.key[i] >= tau ? S.list.mass[i] : 0ull;
    total = block_sum_u64<SB>(total, S.red);
    return total > 0 ? rank_list<false>(S, listed, tau, 0, (double)pp * (double)total) : 0;
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
__device__ __forceinline__ void token_of_tiles(SampleLds& S, const float* row, int V, const Mass& mass, uint32_t tau, float uniform, int last, int amax,
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
        const int at = (tile * m + g0) * 256 + 4 * lane;
        float l[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) l[e] = row[at + e < V ? at + e : V - 1];
        u64 one[4], sum = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            one[e] = at + e < V && okey(l[e]) >= tau ? mass(l[e]) : 0ull;
            sum += one[e];
        }
        u64 in = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const u64 n = __shfl_up(in, o, 64);
            if (lane >= o) in += n;
        }
        votes = __builtin_amdgcn_ballot_w64(sum > 0 && target < (double)(run + in));
        if (votes != 0) {
            if (lane != __builtin_ctzll(votes)) return;
            u64 to = run + in - sum;
            int pick = 3;
#pragma unroll
            for (int e = 0; e < 3; ++e) {   // (the fourth, if none of these: the sum passes the target)
                to += one[e];
                if (pick == 3 && one[e] > 0 && target < (double)to) pick = e;
            }
            *out = at + pick;
            return;
        }
        run += __shfl(in, 63, 64);
    }
    if (lane == 0) *out = last >= 0 ? last : amax;
}

__device__ __forceinline__ void clear_tiles(SampleLds& S, int tiles) {
    __syncthreads();
    for (int t = threadIdx.x; t < tiles; t += SB) S.tile[t] = 0;
    if (threadIdx.x == 0) S.pick = 0;
    __syncthreads();
}

// Adds the list's elements from `tau` on to their tiles; S.pick: the last of them + 1, if it was less
__device__ __forceinline__ void list_to_tiles(SampleLds& S, int listed, uint32_t tau, int m) {
    for (int i = threadIdx.x; i < listed; i += SB)
        if (S.list.key[i] >= tau) {
            atomicAdd(&S.tile[S.list.index[i] / (256 * m)], S.list.mass[i]);
            atomicMax(&S.pick, S.list.index[i] + 1);
        }
    __syncthreads();
}

// Inverse CDF in vocabulary order over the elements of a short list from `tau` on
__device__ __forceinline__ void token_of_list(SampleLds& S, int listed, uint32_t tau, float uniform, int amax, int* out) {
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

// A row by one workgroup.  mx and amax are its maximum; `known`: 1: the top-k's threshold is `tau`, 2: and no top-p is left to be found.
// `per`: bins_per of it.  TIES: a row of ties (sample_of).
template <bool TIES>
__device__ __noinline__ void sample_row(SampleLds& S, const float* row, int V, float mx, int amax, float temp, int k, float pp, float uniform,
                                        int cut, int* out, float per, int known, uint32_t tau) {
    const Mass mass = {mx, 1.0f / temp, cut};
    int listed = -1;    // >= 0: the list holds that many elements, all of the kept ones (keys from tau on) among them

    if (known == 0 && k > 0 && k < V) {
        // threshold of the top-k: the k-th largest key.  The last bin is not counted (under a mask most of a row falls there)
        clear_hist(S);
        over_row<SB>(row, V, [&](int, float l) {
            const int b = bin_of(l, mx, per);
            if (b < NBINS - 1) {
                if (TIES) add_once(&S.hist[b], 1ull, (uint32_t)b);
                else atomicAdd(&S.hist[b], 1ull);
            }
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
    if (known < 2 && pp < 1.0f) {
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
                    if (b == NBINS - 1) rest += m;
                    else if (TIES) add_once(&S.hist[b], m, __float_as_uint(l));
                    else atomicAdd(&S.hist[b], m);
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
                // (a bin of ties has one key, as a rule, which the first of radix_bin's passes finds)
                const int n = TIES ? LIST_CAP + 1
                                   : collect(row, V, S, mass, [&](float l) { return okey(l) >= tau && bin_of(l, mx, per) == bin; });
                tp = n <= LIST_CAP ? rank_list<false>(S, n, tau, base, need) : radix_bin<false>(row, V, S, mass, bin, per, tau, base, need);
            }
        }
        if (!(pp > 0.f)) tp = okey(mx);
        if (tp > tau) tau = tp;
    }
    if (listed >= 0 && listed <= RANK_MAX) {
        token_of_list(S, listed, tau, uniform, amax, out);
        return;
    }
    const int w = threadIdx.x >> 6, m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    int last;
    if (listed >= 0) {
        clear_tiles(S, tiles);
        list_to_tiles(S, listed, tau, m);
        last = S.pick - 1;
    } else {
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
        last = (int)block_max_u32((uint32_t)(my_last + 1), (uint32_t*)S.red) - 1;
    }
    if (w == 0) token_of_tiles(S, row, V, mass, tau, uniform, last, amax, out);
}

// ---- a top-k of few ----------------------------------------------------------------------------------------
// Four threads' elements are a group, whose maxima are distinct elements: the k-th largest of 256 maxima is a bound that at least k
// elements reach, and few more do (of independent numbers 56 for k = 50, 532 for 224).  So the row is read once for the maxima, at one
// instruction an element instead of some 40 for bins, the bound is found by one wave bit by bit in registers, and only threads with an element
// that reaches it read theirs again.  64 rows of 73,448, top-k 50, top-p 0.9: 35 us ->
// 20, top-k 100 25, top-k 200 45 -> 36; 5 rows of 122,753, top-k 50 24, in chunks 26 (46 by one workgroup with histograms).
#define FEW_K 224
#define FEW_GROUPS (SB / 4)
#define FEW_FROM (4 * SB)   // vocabulary from which every thread has elements
#define FEW_WAVE 64       // listed elements that one wave ranks, an element a lane

// Threshold and token of a list of up to 64 elements that holds all of the top-k: by the first wave, an element a lane, each weighed
// against all (rank_list, top_p_of_list and token_of_list in one wave, without their barriers: some 12 us for a list of 60).  Two elements a lane
// lose to the block: 8 rows of 4,096, k 60 15.4 us against 13.3, k 100 21.4 / 16.3, 8 rows of 73,448, k 100 29.2 / 25.0.
__device__ __forceinline__ void token_of_few(const SampleLds& S, int n, int k, float pp, float uniform, int* out) {
    const int lane = threadIdx.x & 63;
    const uint32_t key = lane < n ? S.list.key[lane] : 0u;
    const int index = lane < n ? S.list.index[lane] : -1;
    const u64 mass = lane < n ? S.list.mass[lane] : 0ull;
    int count = 0;
    u64 above = 0;    // mass of the elements with keys from this one's on
#pragma unroll 4
    for (int j = 0; j < n; ++j) {
        const uint32_t kj = S.list.key[j];
        const u64 mj = S.list.mass[j];    // (read whether or not it counts: loads behind a condition wait one after the other)
        count += kj >= key ? 1 : 0;
        above += kj >= key ? mj : 0ull;
    }
    auto largest = [&](uint32_t best) {    // (of a key a lane, or 0)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t v = __shfl_xor(best, o, 64);
            best = v > best ? v : best;
        }
        return best;
    };
    auto kept = [&](uint32_t tau) { return wave_sum_u64(key >= tau ? mass : 0ull); };    // mass of the elements from tau on
    uint32_t tau = largest(count >= k ? key : 0u);
    u64 total = kept(tau);
    if (pp < 1.0f) {
        const double need = (double)pp * (double)total;
        const uint32_t tp = largest(!(pp > 0.f) || (total > 0 && key >= tau && (double)above >= need) ? key : 0u);
        if (tp > tau) {
            tau = tp;
            total = kept(tau);
        }
    }
    const double target = (double)uniform * (double)total;
    u64 run = 0;
#pragma unroll 4
    for (int j = 0; j < n; ++j) {
        const int ij = S.list.index[j];
        const u64 mj = S.list.key[j] >= tau ? S.list.mass[j] : 0ull;
        run += ij <= index ? mj : 0ull;
    }
    // the first index that passes the target (as its complement), else the last kept one
    uint32_t pick = largest(key >= tau && mass > 0 && target < (double)run ? ~(uint32_t)index : 0u);
    if (pick != 0) pick = ~pick;
    else pick = largest(index >= 0 && key >= tau ? (uint32_t)index + 1u : 0u) - 1u;
    if (lane == 0) *out = (int)pick;
}

// The token of a row whose top-k ends in ties: kept are the n listed elements, fewer than k, and all of key `at` below them.  One more reading of the row, an
// instruction or two an element, gives the tiles' masses (5 rows of 122,753 equal numbers, top-p 0.9: 47 us, by histograms 217, in chunks 176)
#define TIE_TILES 8
__device__ __noinline__ void token_of_ties(SampleLds& S, const float* row, int V, Mass mass, uint32_t at, int n, float pp, float uniform, int* out) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    const u64 tie = mass(key_to_float(at));
    const bool whole = ((uintptr_t)row & 15) == 0;
    u64 total = 0;
    for (int t0 = w; t0 < tiles; t0 += TIE_TILES * SNW) {
        int ties[TIE_TILES] = {};
        u64 more[TIE_TILES] = {};
        for (int g = 0; g < m; ++g) {
            float l[TIE_TILES][4];   // of as many tiles at once: a tile's way through memory is longer than its work
#pragma unroll
            for (int u = 0; u < TIE_TILES; ++u) {
                const int i0 = ((t0 + u * SNW) * m + g) * 256 + 4 * lane;
                if (whole && i0 + 3 < V) {
                    const float4 v = *reinterpret_cast<const float4*>(row + i0);
                    l[u][0] = v.x, l[u][1] = v.y, l[u][2] = v.z, l[u][3] = v.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) l[u][e] = row[i0 + e < V ? i0 + e : V - 1];
                }
            }
#pragma unroll
            for (int u = 0; u < TIE_TILES; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool in = ((t0 + u * SNW) * m + g) * 256 + 4 * lane + e < V;
                    const uint32_t key = okey(l[u][e]);
                    ties[u] += __popcll(__builtin_amdgcn_ballot_w64(in && key == at));
                    if (in && key > at && l[u][e] == l[u][e]) more[u] += mass(l[u][e]);
                }
        }
#pragma unroll
        for (int u = 0; u < TIE_TILES; ++u) {
            const int t = t0 + u * SNW;
            if (t >= tiles) break;
            const u64 sum = (u64)ties[u] * tie + (__builtin_amdgcn_ballot_w64(more[u] > 0) != 0ull ? wave_sum_u64(more[u]) : 0ull);
            if (lane == 0) {
                S.tile[t] = sum;
                total += sum;
            }
        }
    }
    uint32_t tau = at;
    if (pp < 1.0f) {
        total = block_sum_u64<SB>(total, S.red);
        const uint32_t tp = pp > 0.f ? rank_list<false>(S, n, 0, 0, (double)pp * (double)total) : okey(mass.mx);
        tau = tp > at ? tp : at;
    }
    if (tau > at) {
        clear_tiles(S, tiles);
        list_to_tiles(S, n, tau, m);
    } else {
        __syncthreads();
    }
    if (w == 0) token_of_tiles(S, row, V, mass, tau, uniform, -1, 0, out);
}

// The row's top-k of 2 to FEW_K; false: the list does not hold it (an infinite maximum with ties, many elements a thread that reach the bound)
__device__ __forceinline__ bool top_k_of_few(SampleLds& S, const float* row, int V, float temp, int k, float pp, float uniform, int cut, int* out) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t* group = reinterpret_cast<uint32_t*>(S.hist);      // [FEW_GROUPS]; behind them the waves' results
    uint32_t* bound = group + FEW_GROUPS;
    float most = -INFINITY;
    over_row<SB>(row, V, [&](int, float l) { most = fmaxf(most, l); });     // (a NaN is dropped)
    float m = fmaxf(most, __shfl_xor(most, 1, 64));
    m = fmaxf(m, __shfl_xor(m, 2, 64));
    if ((lane & 3) == 0) group[threadIdx.x >> 2] = okey(m);
    if (threadIdx.x == 0) S.listed = 0;
    __syncthreads();
    if (w == 0) {
        uint32_t own[FEW_GROUPS / 64], top = 0;
#pragma unroll
        for (int i = 0; i < FEW_GROUPS / 64; ++i) {
            own[i] = group[i * 64 + lane];
            top = own[i] > top ? own[i] : top;
        }
        auto reach = [&](uint32_t at) {
            int n = 0;
#pragma unroll
            for (int i = 0; i < FEW_GROUPS / 64; ++i) n += __popcll(__builtin_amdgcn_ballot_w64(own[i] >= at));
            return n;
        };
        uint32_t at = 0;
#pragma unroll 1
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t c = at | (1u << bit);
            if (reach(c) >= k) at = c;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t v = __shfl_xor(top, o, 64);
            top = v > top ? v : top;
        }
        const int reached = reach(at);    // (by all lanes: behind the branch a ballot counts the first lane's groups alone)
        if (lane == 0) {
            bound[0] = at;
            bound[1] = top;
            bound[2] = (uint32_t)reached;
        }
    }
    __syncthreads();
    const uint32_t at = bound[0];
    const float mx = key_to_float(bound[1]);
    const Mass mass = {mx, 1.0f / temp, cut};
    // Every group at the bound: ties, more perhaps than the list holds (255 of 256 stand for some 1,400 elements where they lie anywhere)
    const bool ties = bound[2] == FEW_GROUPS;
    // At a bound without mass (a mask that leaves fewer than k groups, or a bound far below the maximum) and at one of ties only what lies above is listed:
    // where that comes to fewer than k, the first adds nothing that could be drawn, and the second all of its ties
    const u64 tie = mass(key_to_float(at));
    const bool above = temp > 0.f && mass(mx) > 0 && (ties || tie == 0);
    if (ties && !above) return false;
    const uint32_t least = above ? at + 1 : at;
    if (okey(most) >= least)
        over_row<SB>(row, V, [&](int i, float l) {
            if (okey(l) >= least && l == l) {
                const int to = atomicAdd(&S.listed, 1);
                if (to < LIST_CAP) {
                    S.list.key[to] = okey(l);
                    S.list.index[to] = i;
                    S.list.mass[to] = mass(l);
                }
            }
        });
    __syncthreads();
    const int n = S.listed;
    if (n > LIST_CAP || (n < k && !above)) return false;
    if (n < k && tie > 0) {
        token_of_ties(S, row, V, mass, at, n, pp, uniform, out);
        return true;
    }
    if (n > FEW_WAVE) {
        uint32_t tau = rank_list<true>(S, n, 0, 0, (double)k);
        if (pp < 1.0f) {
            const uint32_t tp = pp > 0.f ? top_p_of_list(S, n, tau, pp) : okey(mx);
            tau = tp > tau ? tp : tau;
        }
        if (n <= RANK_MAX) {
            token_of_list(S, n, tau, uniform, 0, out);
        } else {
            const int g = tile_groups(V);
            clear_tiles(S, (V + 256 * g - 1) / (256 * g));
            list_to_tiles(S, n, tau, g);
            if (w == 0) token_of_tiles(S, row, V, mass, tau, uniform, S.pick - 1, 0, out);
        }
    } else if (w == 0) {
        token_of_few(S, n, k, pp, uniform, out);
    }
    return true;
}

// ---- what each row asks for: in device memory (N 0), or up to N rows' in the launch itself, which saves the copy ahead of it and the buffer that such a
// copy reads.  A kernel's first argument, so it lies where the kernel's arguments begin; read there, as an array among arguments that is
// indexed by the row would be copied into scratch memory first.
template <int N>
struct RowSettings {
    float temperature[N];
    int top_k[N];
    float top_p[N], uniform[N];
};
template <>
struct RowSettings<0> {
    const float* temperature;
    const int* top_k;
    const float *top_p, *uniform;
};
struct Settings {
    float temperature;
    int top_k;
    float top_p, uniform;
};
template <int N>
__device__ __forceinline__ Settings settings_of(const RowSettings<N>& rows, int r) {
    if constexpr (N == 0) {
        return {rows.temperature[r], rows.top_k[r], rows.top_p[r], rows.uniform[r]};
    } else {
        typedef const __attribute__((address_space(4))) RowSettings<N>* Args;
        const Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
        return {a->temperature[r], a->top_k[r], a->top_p[r], a->uniform[r]};
    }
}

template <int N>
__global__ void __launch_bounds__(SB)
sample_kernel(const RowSettings<N> rows, int* __restrict__ out, const float* __restrict__ logits, int V, int stride, int cut) {
    __shared__ SampleLds S;
    const int r = blockIdx.x;
    const Settings set = settings_of<N>(rows, r);
    const int k = set.top_k;
    const float* row = logits + (size_t)r * stride;
    const float temp = set.temperature;
    if (k > 1 && k <= FEW_K && k < V && V >= FEW_FROM && temp != 0.0f && top_k_of_few(S, row, V, temp, k, set.top_p, set.uniform, cut, out + r)) return;
    const RowMax m = block_argmax<SB>(row, V, sample_of(row[(size_t)threadIdx.x * V / SB]), S.meet);
    const float mx = m.value;
    const int amax = m.index == 0x7fffffff ? 0 : m.index;
    if (temp == 0.0f || k == 1) {
        if (threadIdx.x == 0) out[r] = amax;
        return;
    }
    const float per = bins_per(mx, m.seen.low, 1.0f / temp);
    if (m.seen.ties * TIE_SHARE > SB) sample_row<true>(S, row, V, mx, amax, temp, k, set.top_p, set.uniform, cut, out + r, per, 0, 0);
    else sample_row<false>(S, row, V, mx, amax, temp, k, set.top_p, set.uniform, cut, out + r, per, 0, 0);
}

// ---- rows in chunks ----------------------------------------------------------------------------------------
// What a row's chunks leave in the workspace.  The first kernel clears what later ones add to.
struct RowWork {
    u64 hist[NBINS];
    u64 rest;                   // mass of the last bin
    double need;                // the threshold's, as the list's kernel found it: what it has to reach,
    Found found;                // ... its bin,
    int whole;                  // ... and whether the row is left to one workgroup
    int listed, last;           // elements listed; the last element of the bins ahead of the threshold's, + 1
    RowMax max[MAX_CHUNKS];     // of each chunk
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
    __shared__ RowMax meet[CHUNK_THREADS / 64];
    const int r = blockIdx.y;
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    for (int i = blockIdx.x * CHUNK_THREADS + threadIdx.x; i < NBINS; i += gridDim.x * CHUNK_THREADS) W->hist[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        W->rest = 0;
        W->listed = 0;
        W->last = 0;
    }
    const Chunk c = chunk_of(V);
    RowMax m = {-INFINITY, 0x7fffffff, {0, INFINITY}};
    if (c.size > 0) {
        const float* chunk = logits + (size_t)r * stride + c.begin;
        m = block_argmax<CHUNK_THREADS>(chunk, c.size, sample_of(chunk[(size_t)threadIdx.x * c.size / CHUNK_THREADS]), meet);
        if (m.index != 0x7fffffff) m.index += c.begin;
    }
    if (threadIdx.x == 0) W->max[blockIdx.x] = m;
}

// The row's maximum and what its sample tells, a lane a chunk.  `low`: the lowest of the samples of two chunks, the first and one in the
// middle (of all it would be five shuffles more in three kernels)
__device__ __forceinline__ int row_max(const RowWork* W, int chunks, float* mx, bool* ties, float* low) {
    static_assert(MAX_CHUNKS <= 32, "half a wave");
    const int lane = threadIdx.x & 63;
    RowMax m = {-INFINITY, 0x7fffffff, {0, INFINITY}};
    if (lane < chunks) m = W->max[lane];
    const int l = __float_as_int(m.seen.low);
    *low = fminf(__int_as_float(__builtin_amdgcn_readlane(l, 0)), __int_as_float(__builtin_amdgcn_readlane(l, chunks >> 1)));
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
        const float ov = __shfl_xor(m.value, o, 64);
        const int oi = __shfl_xor(m.index, o, 64);
        m.seen.ties += __shfl_xor(m.seen.ties, o, 64);
        better(m.value, m.index, ov, oi);
    }
    const int bi = __builtin_amdgcn_readfirstlane(m.index);
    *mx = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(m.value)));
    *ties = __builtin_amdgcn_readfirstlane(m.seen.ties) * TIE_SHARE > chunks * CHUNK_THREADS;
    return bi == 0x7fffffff ? 0 : bi;
}

template <int N>
__global__ void __launch_bounds__(CHUNK_THREADS)
sample_hist_kernel(const RowSettings<N> rows, char* __restrict__ ws, size_t ws_row, const float* __restrict__ logits, int V, int stride, int cut) {
    __shared__ u64 hist[NBINS];
    __shared__ u64 red[CHUNK_THREADS / 64];
    const int r = blockIdx.y;
    const Settings set = settings_of<N>(rows, r);
    const int k = set.top_k;
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float temp = set.temperature, pp = set.top_p;
    const bool count = k > 0 && k < V;
    if (temp == 0.0f || k == 1 || (!count && !(pp < 1.0f))) return;
    float mx, low;
    bool ties;
    row_max(W, gridDim.x, &mx, &ties, &low);
    const Mass mass = {mx, 1.0f / temp, cut};
    const float per = bins_per(mx, low, mass.inv_t);
    for (int i = threadIdx.x; i < NBINS; i += CHUNK_THREADS) hist[i] = 0;
    __syncthreads();
    const Chunk c = chunk_of(V);
    u64 rest = 0;
    auto fill = [&](auto tied) {
        over_row<CHUNK_THREADS>(logits + (size_t)r * stride + c.begin, c.size, [&](int, float l) {
            const int b = bin_of(l, mx, per);
            const u64 w = count ? 1ull : mass(l);
            if (b == NBINS - 1) rest += w;
            else if (tied) add_once(&hist[b], w, __float_as_uint(l));
            else atomicAdd(&hist[b], w);
        });
    };
    if (ties) fill(std::true_type());
    else fill(std::false_type());
    rest = block_sum_u64<CHUNK_THREADS>(rest, red);   // (its barriers close the histogram too)
    for (int i = threadIdx.x; i < NBINS; i += CHUNK_THREADS)
        if (hist[i] != 0) atomicAdd(&W->hist[i], hist[i]);
    if (threadIdx.x == 0 && rest != 0) atomicAdd(&W->rest, rest);
}

// Where the row's first threshold lies, from its histogram: found.at < 0 and no top-k or top-p: everything is kept; `whole`: the row
// is left to one workgroup (a threshold in the last bin, a top-k beyond the list, no mass, p not above 0).  `mine`: a thread's bins; their
// scan gives the row's mass, by which a top-p's threshold is known, and then its bin.
template <int NT>
__device__ __forceinline__ Found row_threshold(const u64 (&mine)[NBINS / NT], u64 rest, u64* red, Found* shared, bool count, int k, float pp, bool* whole,
                                               double* need) {
    constexpr int PER = NBINS / NT;
    Found f = {-1, 0, 0};
    *whole = false;
    *need = 0;
    if (!count && !(pp < 1.0f)) return f;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u64 sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) sum += mine[i];
    u64 incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 n = __shfl_up(incl, o, 64);
        if (lane >= o) incl += n;
    }
    if (lane == 63) red[w] = incl;
    if (threadIdx.x == 0) *shared = f;
    __syncthreads();
    u64 run = incl - sum, total = rest;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        const u64 v = red[i];
        if (i < w) run += v;
        total += v;
    }
    *need = count ? (double)k : (double)pp * (double)total;
    if (!count && (!(pp > 0.f) || total == 0)) {
        *whole = true;
        return f;
    }
    if (!((double)run >= *need)) {   // (not reached before this thread's entries)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!((double)run >= *need) && (double)(run + mine[i]) >= *need) *shared = {(int)threadIdx.x * PER + i, run, mine[i]};
            run += mine[i];
        }
    }
    __syncthreads();
    f = *shared;
    *whole = f.at < 0 || (count && f.before + f.in > LIST_CAP);
    return f;
}

template <int N>
__global__ void __launch_bounds__(CHUNK_THREADS)
sample_list_kernel(const RowSettings<N> rows, char* __restrict__ ws, size_t ws_row, const float* __restrict__ logits, int V, int stride, int cut) {
    __shared__ u64 red[CHUNK_THREADS / 64];
    __shared__ Found shared;
    __shared__ uint32_t keys[LIST_CAP];   // the chunk's listed elements: a place in the row's list costs a round trip through memory, so a chunk asks
    __shared__ int indices[LIST_CAP];     // once for all of its own
    __shared__ int own, from, last;
    const int r = blockIdx.y;
    const Settings set = settings_of<N>(rows, r);
    const int k = set.top_k;
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float* row = logits + (size_t)r * stride;
    const float temp = set.temperature, pp = set.top_p;
    const bool count = k > 0 && k < V;
    if (temp == 0.0f || k == 1) return;
    if (threadIdx.x == 0) own = 0, last = 0;
    // what the kernel reads is on its way at once: the bins, the chunks' maxima, and a wave's first two tiles
    u64 mine[NBINS / CHUNK_THREADS];
#pragma unroll
    for (int i = 0; i < NBINS / CHUNK_THREADS; ++i) mine[i] = W->hist[threadIdx.x * (NBINS / CHUNK_THREADS) + i];
    const u64 rest = W->rest;
    const Chunk c = chunk_of(V);
    const int m = tile_groups(V), t0 = c.first + (int)(threadIdx.x >> 6), lane4 = 4 * (int)(threadIdx.x & 63);
    float ahead[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = (t0 + u * (CHUNK_THREADS / 64)) * 256 + lane4 + e;
            ahead[u][e] = row[i < V ? i : V - 1];
        }
    float mx, low;
    bool ties;
    row_max(W, gridDim.x, &mx, &ties, &low);
    bool whole;
    double need;
    const Found f = row_threshold<CHUNK_THREADS>(mine, rest, red, &shared, count, k, pp, &whole, &need);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        W->need = need;
        W->found = f;
        W->whole = whole ? 1 : 0;
    }
    if (whole) return;
    const Mass mass = {mx, 1.0f / temp, cut};
    const float per = bins_per(mx, low, mass.inv_t);
    __syncthreads();   // (`own`)
    auto list = [&](int i, float l) {
        const int at = atomicAdd(&own, 1);
        if (at < LIST_CAP) {
            keys[at] = okey(l);
            indices[at] = i;
        }
    };
    if (count) {   // everything down to the threshold's bin
        over_row<CHUNK_THREADS>(row + c.begin, c.size, [&](int i, float l) {
            if (bin_of(l, mx, per) <= f.at) list(c.begin + i, l);
        });
    } else {
        const int above = f.at >= 0 ? f.at : NBINS;   // the bins ahead of the threshold's are kept whole
        int my_last = -1;
        auto tile = [&](int t, auto over) {
            u64 sum = 0;
            over([&](int i, float l) {
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
        };
        int t = t0;
        if (m == 1) {
#pragma unroll
            for (int u = 0; u < 2; ++u, t += CHUNK_THREADS / 64)
                if (t < c.first + c.count)
                    tile(t, [&](auto f) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (t * 256 + lane4 + e < V) f(t * 256 + lane4 + e, ahead[u][e]);
                    });
        }
        for (; t < c.first + c.count; t += CHUNK_THREADS / 64) tile(t, [&](auto f) { over_tile(row, V, t, m, f); });
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const int v = __shfl_xor(my_last, o, 64);
            my_last = v > my_last ? v : my_last;
        }
        if ((threadIdx.x & 63) == 0) atomicMax(&last, my_last + 1);
    }
    __syncthreads();
    if (threadIdx.x == 0 && last != 0) atomicMax(&W->last, last);   // (an atomic a chunk: one of every thread held the row's address for half the kernel)
    const int n = own;
    if (n == 0) return;
    if (threadIdx.x == 0) from = atomicAdd(&W->listed, n);
    __syncthreads();
    for (int i = threadIdx.x; i < n && i < LIST_CAP && from + i < LIST_CAP; i += CHUNK_THREADS) {
        W->key[from + i] = keys[i];
        W->index[from + i] = indices[i];
    }
}

template <int N>
__global__ void __launch_bounds__(SB)
sample_token_kernel(const RowSettings<N> rows, int* __restrict__ out, char* __restrict__ ws, size_t ws_row, int chunks, const float* __restrict__ logits,
                    int V, int stride, int cut) {
    __shared__ SampleLds S;
    const int r = blockIdx.x;
    const Settings set = settings_of<N>(rows, r);
    const int k = set.top_k;
    RowWork* W = reinterpret_cast<RowWork*>(ws + (size_t)r * ws_row);
    const float* row = logits + (size_t)r * stride;
    const float temp = set.temperature, pp = set.top_p;
    const bool count = k > 0 && k < V;
    float mx, low;
    bool ties;
    const int amax = row_max(W, chunks, &mx, &ties, &low);
    if (temp == 0.0f || k == 1) {
        if (threadIdx.x == 0) out[r] = amax;
        return;
    }
    const Found f = W->found;
    const double need = W->need;
    const int listed = W->listed;
    const Mass mass = {mx, 1.0f / temp, cut};
    if (W->whole != 0 || listed > LIST_CAP) {
        uint32_t tau = 0;
        int known = 0;
        const float per = bins_per(mx, low, mass.inv_t);
        if (f.at >= 0) {   // the threshold's bin is known, the list does not hold it
            known = count ? 1 : 2;
            tau = count ? radix_bin<true>(row, V, S, mass, f.at, per, 0, f.before, need)
                        : radix_bin<false>(row, V, S, mass, f.at, per, 0, f.before, need);
        }
        if (ties) sample_row<true>(S, row, V, mx, amax, temp, k, pp, set.uniform, cut, out + r, per, known, tau);
        else sample_row<false>(S, row, V, mx, amax, temp, k, pp, set.uniform, cut, out + r, per, known, tau);
        return;
    }
    for (int i = threadIdx.x; i < listed; i += SB) {
        const uint32_t key = W->key[i];
        S.list.key[i] = key;
        S.list.index[i] = W->index[i];
        S.list.mass[i] = mass(key_to_float(key));
    }
    const int m = tile_groups(V), tiles = (V + 256 * m - 1) / (256 * m);
    if (!count) {
        for (int t = threadIdx.x; t < tiles; t += SB) S.tile[t] = W->tile[t];
        if (threadIdx.x == 0) S.pick = W->last;
    }
    __syncthreads();
    uint32_t tau = 0;
    if (count) {
        tau = rank_list<true>(S, listed, 0, 0, need);
        if (pp < 1.0f) {
            const uint32_t tp = pp > 0.f ? top_p_of_list(S, listed, tau, pp) : okey(mx);
            if (tp > tau) tau = tp;
        }
        if (listed <= RANK_MAX) {
            token_of_list(S, listed, tau, set.uniform, amax, out + r);
            return;
        }
        clear_tiles(S, tiles);
    } else {
        if (f.at >= 0) tau = rank_bin(S, listed, 0, f.before, need);
    }
    list_to_tiles(S, listed, tau, m);
    if (threadIdx.x < 64) token_of_tiles(S, row, V, mass, tau, set.uniform, S.pick - 1, amax, out + r);
}

// Bytes of workspace a row needs of n rows of V logits; 0: none, the rows are not cut into chunks.  They are where few rows leave
// the chip idle and a row is long enough to outweigh three more launches.  In chunks against one workgroup a row, us, with top-p
// alone, with top-k 50 and with neither (which of them rows ask for is only known on the device):
//   32,768:  1 row 31 / 37, 26 / 15, 18 / 20;  8 rows 34 / 38, 28 / 17, 18 / 20;  32 rows 36 / 38, 30 / 17, 19 / 20  (chunks: before their
//            kernels were made shorter)
//   49,152:  8 rows 27 / 49, 26 / 17, 17 / 26;  32 rows 32 / 50, 31 / 18, 20 / 26;  64 rows 47 / 52, 36 / 18, 24 / 28
//   73,448:  1 row 26 / 65, 24 / 19, 17 / 34;  32 rows 39 / 68, 35 / 20, 22 / 35;  64 rows 55 / 69, 42 / 20, 29 / 36
//   122,753: 5 rows 30 / 103, 26 / 24, 17 / 56;  32 rows 45 / 105, 41 / 25, 25 / 56;  64 rows 53 / 111, 43 / 27, 32 / 62;
//            96 rows 80 / 115, 55 / 29, 43 / 63
// A caller who knows that every row asks for a top-k of at most FEW_K may give no workspace and have them by one workgroup each (the rule: kernels.sample_one_reading).
#define CHUNKS_FROM 40960
#define CHUNKS_MANY_FROM 98304      // ... with more than 32 rows, up to 64
extern "C" long ilm_sample_ws(int n, int V) {
    if (V <= CHUNKS_FROM || n > (V > CHUNKS_MANY_FROM ? 64 : 32)) return 0;
    return (long)(sizeof(RowWork) + sizeof(u64) * ((V + 255) / 256) + 15) / 16 * 16;
}

// The largest top-k that a row is served with in one reading (top_k_of_few)
extern "C" int ilm_sample_few_k() { return FEW_K; }

static inline uint64_t mix64(uint64_t x) {   // splitmix64's finaliser
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D2049BB133111Bull;
    return x ^ (x >> 31);
}

// On the host: out[i] = the uniform number of (seeds[i], keys[i], indices[i]), n of each; `seeds` null: `seed` for all
extern "C" int ilm_uniforms(float* out, const uint64_t* seeds, uint64_t seed, const uint64_t* keys, const uint64_t* indices, int n) {
    ILM_REQUIRE(n >= 0 && (n == 0 || (out != nullptr && keys != nullptr && indices != nullptr)), "uniforms: bad arguments, n=%d", n);
    for (int i = 0; i < n; ++i) {
        const uint64_t x = mix64(mix64(mix64(seeds != nullptr ? seeds[i] : seed) ^ keys[i]) ^ indices[i]);
        out[i] = (float)(x >> 40) / 16777216.0f;
    }
    return 0;
}

template <int N>
static int sample_rows(const RowSettings<N>& rows, void* out, const void* logits, void* ws, int n, int V, int stride, hipStream_t stream) {
    int cut = 0;   // V elements of at most 2^43 each: below 2^64 up to a vocabulary of 2^20
    while ((long long)V >> (20 + cut)) ++cut;
    const size_t ws_row = (size_t)ilm_sample_ws(n, V);
    if (ws == nullptr || ws_row == 0) {
        sample_kernel<N><<<n, SB, 0, stream>>>(rows, (int*)out, (const float*)logits, V, stride, cut);
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
    sample_hist_kernel<N><<<grid, CHUNK_THREADS, 0, stream>>>(rows, w, ws_row, (const float*)logits, V, stride, cut);
    sample_list_kernel<N><<<grid, CHUNK_THREADS, 0, stream>>>(rows, w, ws_row, (const float*)logits, V, stride, cut);
    sample_token_kernel<N><<<n, SB, 0, stream>>>(rows, (int*)out, w, ws_row, chunks, (const float*)logits, V, stride, cut);
    ILM_LAUNCH_CHECK("sample");
    return 0;
}
static int sample_check(int n, int V, int stride, const void* ws) {
    ILM_REQUIRE(n > 0 && V > 0 && stride >= V, "sample: bad sizes n=%d V=%d stride=%d", n, V, stride);
    ILM_REQUIRE(((uintptr_t)ws & 15) == 0, "sample: the workspace must be 16-byte aligned");
    return 0;
}

// `ws`: n * ilm_sample_ws(n, V) bytes, 16-byte aligned, or null: every row by one workgroup
extern "C" int ilm_sample(void* out, const void* logits, const void* temperature, const void* top_k,
                          const void* top_p, const void* uniform, void* ws, int n, int V, int stride,
                          hipStream_t stream) {
    if (sample_check(n, V, stride, ws) != 0) return -1;
    const RowSettings<0> rows = {(const float*)temperature, (const int*)top_k, (const float*)top_p, (const float*)uniform};
    return sample_rows<0>(rows, out, logits, ws, n, V, stride, stream);
}

// The same with what the rows ask for at host addresses, read before the call returns (a recorded call keeps it), for up to ilm_sample_host_rows() rows;
// the uniform numbers from seeds (null: `seed` for all), keys and indices as ilm_uniforms forms them.  64 rows of 73,448 with a top-k of 50 through the
// sampler 32.7 -> 21.6 us a call, 5 of 122,753 with top-p 35.9 -> 29.5 (a copy of 2 us and what waits for it less, and 12 us less on the host).
extern "C" int ilm_sample_host_rows() { return 192; }   // (16 bytes a row, within the 4 KB that a launch's arguments may take)
extern "C" int ilm_sample_host(void* out, const void* logits, const float* temperature, const int* top_k, const float* top_p, const uint64_t* seeds,
                               uint64_t seed, const uint64_t* keys, const uint64_t* indices, void* ws, int n, int V, int stride, hipStream_t stream) {
    if (sample_check(n, V, stride, ws) != 0) return -1;
    ILM_REQUIRE(n <= ilm_sample_host_rows(), "sample_host: %d rows", n);
#define SAMPLE_HOST(N_)                                                                        \
    {                                                                                          \
        RowSettings<N_> rows;                                                                  \
        memcpy(rows.temperature, temperature, n * sizeof(float));                              \
        memcpy(rows.top_k, top_k, n * sizeof(int));                                            \
        memcpy(rows.top_p, top_p, n * sizeof(float));                                          \
        if (ilm_uniforms(rows.uniform, seeds, seed, keys, indices, n) != 0) return -1;         \
        return sample_rows<N_>(rows, out, logits, ws, n, V, stride, stream);                   \
    }
    if (n <= 16) SAMPLE_HOST(16)
    if (n <= 64) SAMPLE_HOST(64)
    SAMPLE_HOST(192)
#undef SAMPLE_HOST
}
