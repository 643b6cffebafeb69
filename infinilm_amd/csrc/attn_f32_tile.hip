// Paged attention of the 32-bit path for runs of consecutive tokens of a request (portions of prompts): the sums of attn_f32.hip
// in the same order, so a token has the same bits here and alone, with the keys read once for up to eight tokens.
//
// What bounds it: the float matrix instruction (32 cycles for 16 x 16 x 4; 157 TFLOP/s nominal over the chip).  A wave that takes its
// token's keys from memory by itself, 16 rows of 64 bytes an instruction, is bound by that instead.  Here a workgroup takes a tile of up to
// eight tokens and one KV head's query heads, and keys and values go through LDS (`global_load_lds`, no registers on the way) in two stages, one
// on its way, for all of its waves.  The columns of the matrix instruction are (token, head) pairs: one token of 9 to 16 heads
// a wave, two of 5 to 8, four of 3 or 4, eight of one or two (a head alone would leave 15 of 16 columns idle).
//
// Measured, tokens one by one before and in tiles now: 2,048 tokens of 32 heads of 128 over 2 KV heads 660 -> 404 us (the matrix cores busy 0.6 of
// the time, the rest exponentials and the ends of workgroups), of 32 over 8 2,010 -> 398, of 36 heads of 64 over 36 4,220 -> 541, of 16 of 64 over
// 2 346 -> 180; 300 of 32 over 2 38 -> 34.  Two workgroups of four tokens a tile where a wave takes one: one of eight 420, whose waves meet the
// exponentials at once.  Two stages of 64 keys in LDS: four of 32 449.  Scores of two tiles of keys side by side, and pages looked up by a shift.
// A wave that multiplies goes ahead of one at its exponentials (s_setprio): 404 -> 377, 180 -> 147.
//
// Rows lie in LDS so that the 16 rows of an operand fall on distinct banks: the 16-byte pieces of a key's row are exchanged by the
// row's number, those of a dim's 16 keys (64 bytes) by its half of eight rows; the exchange is made on the source side of the load.
#include "attn_f32.h"

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef const __attribute__((address_space(4))) int* const_ints;   // (read by the scalar unit whatever stands in between)

// DT: head size / 16; NW: waves, of TPW tokens each
template <int DT, int NW>
struct FtShape {
    static constexpr int S = NW == 4 ? 4 : 2;   // tiles of 16 keys a stage
    static constexpr int RING = 2;              // stages in LDS
    static constexpr int BLOCKS = S * DT, EACH = DT / NW;   // loads of 1 KB a stage; of a tile and a wave
    static_assert(DT % NW == 0 && FA_TILES % S == 0, "whole loads");
};

// SPLIT: blockIdx.z is the chunk, whose partial result goes to ws (attn_f32.h: the rows of the tile's eight); else a workgroup walks all chunks of its tokens.
template <int DT, int NW, int TPW, bool SPLIT>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2)))
attn_f32_tile_kernel(float* __restrict__ out, float* __restrict__ ws, const float* __restrict__ qp, const float* __restrict__ kc, const float* __restrict__ vc,
                     const int* __restrict__ block_tables, const int* __restrict__ seg, const int* __restrict__ pos,
                     const int* __restrict__ tiles, int n_tiles, int nh, int nkv, int nsub, int page, int shift, int max_blocks, int q_stride,
                     int out_stride, float scale, int reach, float softcap) {
    typedef FtShape<DT, NW> Sh;
    constexpr int d = DT * 16, S = Sh::S, RING = Sh::RING, EACH = Sh::EACH, HW = 16 / TPW, STAGES = FA_TILES / S;
    __shared__ __align__(16) float4 lds[RING][Sh::BLOCKS * 64];
    // the longest tiles first: they stand last in the list
    const int tile = n_tiles - 1 - (int)blockIdx.y;
    // the tile's part of NW x TPW tokens (the later part of the same keys first)
    const int part = FT_TOKENS - NW * TPW - (int)(blockIdx.x / (nkv * nsub)) * (NW * TPW);
    const int row0 = tiles[2 * tile] + part, in_tile = tiles[2 * tile + 1], count = min(in_tile - part, NW * TPW);
    if (in_tile < 0 && (!SPLIT || blockIdx.z == 0)) {   // rows of no request get zeros
        const int G = nh / nkv, kvh = blockIdx.x / nsub % nkv, sub = blockIdx.x % nsub, of_row = min(16, G - sub * 16) * (d / 4);
        const int n = min(-in_tile - part, NW * TPW) * of_row;
        float* from = out + (size_t)row0 * out_stride + (size_t)(kvh * G + sub * 16) * d;
        for (int i = threadIdx.x; i < n; i += NW * 64) reinterpret_cast<float4*>(from + (size_t)(i / of_row) * out_stride)[i % of_row] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (count <= 0) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int G = nh / nkv, kvh = blockIdx.x / nsub % nkv, sub = blockIdx.x % nsub;
    const int heads = (G - sub * 16 < HW) ? G - sub * 16 : HW;
    const int h = kvh * G + sub * 16 + (r % HW < heads ? r % HW : heads - 1);
    const bool live = wave * TPW + r / HW < count && r % HW < heads;
    auto row_of = [&](int i) { return row0 + (i < count ? i : count - 1); };
    const int t = row_of(wave * TPW + r / HW);
    const int p = pos[t], lo = first_key(p, reach);
    // first and last position of the workgroup's tokens and of the wave's
    const const_ints cpos = (const_ints)(uintptr_t)pos;
    const int p_first = cpos[row0], p_last = cpos[row_of(NW * TPW)], lo_first = first_key(p_first, reach);
    const int pw_last = cpos[row_of(wave * TPW + TPW - 1)], low_first = first_key(cpos[row_of(wave * TPW)], reach);
    const int pw_first = cpos[row_of(wave * TPW)], low_last = first_key(pw_last, reach);
    const int c_first = SPLIT ? (int)blockIdx.z : lo_first / FA_CHUNK, c_last = SPLIT ? (int)blockIdx.z : p_last / FA_CHUNK;
    if (SPLIT && (c_first < lo_first / FA_CHUNK || c_last > p_last / FA_CHUNK)) return;   // (the fold reads only the chunks a token sees)
    const bool wave_live = wave * TPW < count;
    const const_ints bt = (const_ints)(uintptr_t)(block_tables + (size_t)((const_ints)(uintptr_t)seg)[row0] * max_blocks);

    float4 qf[DT];
    {
        const float4* qrow = reinterpret_cast<const float4*>(qp + (size_t)t * q_stride + (size_t)h * d);
#pragma unroll
        for (int j = 0; j < DT; ++j) qf[j] = qrow[4 * j + q];
    }

    // ---- the stages: of a chunk its tiles' keys, then their values, chunk after chunk
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)(&lds[0][0]);
    // in bytes: the lane's 16 of a load, from the tile's first key (its place of dim 0) on; for values by what differs from the keys' (a select
    // between the two arrays became an index into scratch memory)
    uint32_t koff[EACH], kv_xor[EACH];
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        const int j = wave + NW * i, at = j * 64 + lane, row = at / (4 * DT), slot = at % (4 * DT);
        koff[i] = (uint32_t)(row * d + ((slot ^ row) * 4)) * 4u;
        const int vrow = lane >> 2;
        kv_xor[i] = koff[i] ^ (((uint32_t)(16 * j + vrow) * (uint32_t)page + (((lane & 3) ^ ((vrow >> 3) * 3)) * 4)) * 4u);
    }
    auto first_tile = [&](int c) { return lo_first > c * FA_CHUNK ? (lo_first - c * FA_CHUNK) >> 4 : 0; };
    auto last_tile = [&](int c) { return p_last < c * FA_CHUNK + FA_CHUNK - 1 ? (p_last - c * FA_CHUNK) >> 4 : FA_TILES - 1; };
    int pc = c_first, pv = 0, ps = first_tile(c_first) / S, pbuf = 0;   // the stage to be asked for next: chunk, values or keys, number; its buffer
    int pg[S], at[S];                                                   // ... its tiles' pages and places in them
    auto look_up = [&]() {
        const int ta = first_tile(pc), tb = last_tile(pc);
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int kt = ps * S + u, base = pc * FA_CHUNK + 16 * (kt < ta ? ta : (kt > tb ? tb : kt));
            const int b = shift >= 0 ? base >> shift : base / page;
            at[u] = base - b * page;
            pg[u] = bt[b];
        }
    };
    auto issue = [&]() {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const size_t head = (size_t)pg[u] * nkv + kvh;
            const float* from = pv ? vc + head * d * page + at[u] : kc + (head * page + at[u]) * d;
#pragma unroll
            for (int i = 0; i < EACH; ++i)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(
                                 lds0 + (uint32_t)((pbuf * Sh::BLOCKS + u * DT + wave + NW * i) * 1024)),
                             "v"(koff[i] ^ (kv_xor[i] & (uint32_t)-pv)), "s"(from)
                             : "m0", "memory");
        }
        pbuf = pbuf + 1 == RING ? 0 : pbuf + 1;
        if (ps < last_tile(pc) / S) {
            ++ps;
        } else if (!pv) {
            pv = 1;
            ps = first_tile(pc) / S;
        } else if (pc < c_last) {
            ++pc;
            pv = 0;
            ps = first_tile(pc) / S;
        }   // else: the last stage again, so that the waits can count
        look_up();
    };
    look_up();
#pragma unroll
    for (int i = 0; i < RING - 1; ++i) issue();
    int buf = 0;
    auto take = [&]() {   // the next stage in order: its loads have landed, everybody's, and everybody is done with the one before
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((RING - 2) * S * EACH) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue();
        const float4* at_ = lds[buf];
        buf = buf + 1 == RING ? 0 : buf + 1;
        return at_;
    };

    float M = -INFINITY, L = 0.f;
    f32x4 ACC[SPLIT ? 1 : DT];
#pragma unroll
    for (int i = 0; i < (SPLIT ? 1 : DT); ++i) ACC[i] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll 1
    for (int c = c_first; c <= c_last; ++c) {
        const int c0 = c * FA_CHUNK, sa = first_tile(c) / S, sb = last_tile(c) / S;
        const int k_lo = lo > c0 ? lo : c0, k_hi = p < c0 + FA_CHUNK - 1 ? p : c0 + FA_CHUNK - 1;   // what the column's token sees
        const bool sees = k_lo <= k_hi;
        // tiles with a key that some token of the wave sees, and (in between) those that all of them see whole
        const bool any = wave_live && pw_last >= c0 && low_first < c0 + FA_CHUNK;
        const int wa = any ? (low_first > c0 ? (low_first - c0) >> 4 : 0) : FA_TILES;
        const int wb = any ? (pw_last < c0 + FA_CHUNK - 1 ? (pw_last - c0) >> 4 : FA_TILES - 1) : -1;
        auto whole = [&](int kt) { return c0 + 16 * kt >= low_last && c0 + 16 * kt + 15 <= pw_first; };

        // ---- scores
        __builtin_amdgcn_s_setprio(1);
        f32x4 Sc[FA_TILES];
#pragma unroll
        for (int sg = 0; sg < STAGES; ++sg) {
            if (sg < sa || sg > sb) {
#pragma unroll
                for (int u = 0; u < S; ++u) Sc[sg * S + u] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                continue;
            }
            const float4* keys = take();
#pragma unroll
            for (int u = 0; u < S; u += 2) {   // (two chains of products side by side)
                const int kt = sg * S + u;
                Sc[kt] = Sc[kt + 1] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                if (kt + 1 < wa || kt > wb) continue;
                const float4* krow = keys + u * (64 * DT) + r * (4 * DT);
                f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                for (int j = 0; j < DT; ++j) {
                    const float4 k0 = krow[(4 * j + q) ^ r], k1 = krow[64 * DT + ((4 * j + q) ^ r)];
                    s[0] = fa_mfma(k0.x, qf[j].x, s[0]);
                    s[1] = fa_mfma(k1.x, qf[j].x, s[1]);
                    s[0] = fa_mfma(k0.y, qf[j].y, s[0]);
                    s[1] = fa_mfma(k1.y, qf[j].y, s[1]);
                    s[0] = fa_mfma(k0.z, qf[j].z, s[0]);
                    s[1] = fa_mfma(k1.z, qf[j].z, s[1]);
                    s[0] = fa_mfma(k0.w, qf[j].w, s[0]);
                    s[1] = fa_mfma(k1.w, qf[j].w, s[1]);
                }
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const int key0 = c0 + (kt + v) * 16 + 4 * q;   // element e is the score of key key0 + e
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float sc = s[v][e] * scale;
                        if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
                        Sc[kt + v][e] = (key0 + e >= k_lo && key0 + e <= k_hi) ? sc : -INFINITY;
                    }
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        // ---- maximum, exponentials and their sum per column, which lies in the four lanes r, r + 16, r + 32, r + 48
        float m = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < FA_TILES; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = fmaxf(m, Sc[kt][e]);
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        const float ref = sees ? m : 0.f;   // (a column that sees none of the chunk has weights of zero)
        float l = 0.f;
#pragma unroll
        for (int kt = 0; kt < FA_TILES; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                Sc[kt][e] = expf(Sc[kt][e] - ref);
                l += Sc[kt][e];
            }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);

        // ---- weighted values
        __builtin_amdgcn_s_setprio(1);
        f32x4 acc[DT];
#pragma unroll
        for (int i = 0; i < DT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int sg = 0; sg < STAGES; ++sg) {
            if (sg < sa || sg > sb) continue;
            const float4* values = take();
#pragma unroll
            for (int u = 0; u < S; ++u) {
                const int kt = sg * S + u;
                if (kt < wa || kt > wb) continue;
                const float4* vrow = values + u * (64 * DT) + r * 4 + (q ^ ((r >> 3) * 3));
                const f32x4 w = Sc[kt];
                if (whole(kt)) {
#pragma unroll
                    for (int i = 0; i < DT; ++i) {
                        const float4 v = vrow[i * 64];
                        acc[i] = fa_mfma(v.x, w[0], acc[i]);
                        acc[i] = fa_mfma(v.y, w[1], acc[i]);
                        acc[i] = fa_mfma(v.z, w[2], acc[i]);
                        acc[i] = fa_mfma(v.w, w[3], acc[i]);
                    }
                    continue;
                }
                // An edge.  Values that none of the wave's tokens sees may be anything (pages are not cleared) and count as zeros; those that only
                // some see have weights of zero in the others' columns, which is enough unless one is not finite: then a token at a time
                const int key0 = c0 + kt * 16 + 4 * q;
                auto mul = [&](const f32x4 (&from)[DT], int a, int b, auto&& keep) {
#pragma unroll
                    for (int i = 0; i < DT; ++i) {
                        const float4 v = vrow[i * 64];
                        f32x4 s = from[i];
                        s = fa_mfma(key0 >= a && key0 <= b ? v.x : 0.f, w[0], s);
                        s = fa_mfma(key0 + 1 >= a && key0 + 1 <= b ? v.y : 0.f, w[1], s);
                        s = fa_mfma(key0 + 2 >= a && key0 + 2 <= b ? v.z : 0.f, w[2], s);
                        s = fa_mfma(key0 + 3 >= a && key0 + 3 <= b ? v.w : 0.f, w[3], s);
                        keep(i, s);
                    }
                };
                bool odd = false;
                if (TPW > 1) {
                    auto bad = [&](float v, int e) { return key0 + e >= low_first && key0 + e <= pw_last && !(fabsf(v) <= 3.402823466e38f); };
#pragma unroll
                    for (int i = 0; i < DT; ++i) {
                        const float4 v = vrow[i * 64];
                        odd = odd || bad(v.x, 0) || bad(v.y, 1) || bad(v.z, 2) || bad(v.w, 3);
                    }
                }
                if (TPW == 1 || __builtin_amdgcn_ballot_w64(odd) == 0ull) {
                    mul(acc, low_first, pw_last, [&](int i, const f32x4& s) { acc[i] = s; });
                } else {
#pragma unroll 1
                    for (int tok = 0; tok < TPW; ++tok) {
                        const int pt = cpos[row_of(wave * TPW + tok)];
                        const bool own = r / HW == tok;
                        mul(acc, first_key(pt, reach), pt, [&](int i, const f32x4& s) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][e] = own ? s[e] : acc[i][e];
                        });
                    }
                }
            }
        }
        if (SPLIT) {
            if (live && sees) {
                float* dst = ws + (((size_t)(tile * FT_TOKENS + part + wave * TPW + r / HW) * nh + h) * gridDim.z + c) * (d + FA_WS_PAD);
#pragma unroll
                for (int i = 0; i < DT; ++i) *reinterpret_cast<f32x4*>(dst + 16 * i + 4 * q) = acc[i];
                if (q == 0) {
                    dst[d] = m;
                    dst[d + 1] = l;
                }
            }
            continue;
        }
        float Mn = M, Ln = L, a, b;
        fa_fold_scales(Mn, Ln, m, l, a, b);
        M = sees ? Mn : M;
        L = sees ? Ln : L;
        a = sees ? a : 1.f;
        b = sees ? b : 0.f;
#pragma unroll
        for (int i = 0; i < (SPLIT ? 0 : DT); ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) ACC[i][e] = fmaf(ACC[i][e], a, acc[i][e] * b);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the loads beyond the last stage: LDS is handed on when the workgroup ends)
    if (!SPLIT && live) {
        float* orow = out + (size_t)t * out_stride + (size_t)h * d;
        const float inv = 1.0f / L;
#pragma unroll
        for (int i = 0; i < (SPLIT ? 0 : DT); ++i) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = ACC[i][e] * inv;
            *reinterpret_cast<f32x4*>(orow + 16 * i + 4 * q) = o;
        }
    }
}

// Whether the tile form takes such heads and pages (offsets inside a page take 32 bits).  Heads: the exchange of a row's pieces of 16 bytes wants a power of two of
// at least 16 of them, which leaves out 32, 80, 96 and 192; 256, with twice the queries and sums in registers and twice the LDS a stage, was not built.
extern "C" int ilm_attn_f32_tile_ok(int d, int page) {
    return (d == 64 || d == 128) && page > 0 && page % 16 == 0 && (long long)d * page < (1ll << 28) ? 1 : 0;
}
extern "C" int ilm_attn_f32_tile_tokens() { return FT_TOKENS; }

// tiles: n_tiles pairs (first row, count <= 8; 0: nothing; below 0: that many rows of no request) of rows of consecutive tokens of one request;
// rows of `out` that no tile holds are left alone.
// ws: null, or float [8 n_tiles][nh][nchunks][d + 4] (as ilm_attn_f32): a workgroup a chunk, and with `fold` the fold of them; without, that is left to the
// call for the step's single tokens.
extern "C" int ilm_attn_f32_tile(void* out, void* ws, int nchunks, const void* q, const void* kc, const void* vc, const void* block_tables, const void* seg, const void* pos,
                                 const void* tiles, int n_tiles, int fold, int nh, int nkv, int d, int page, int max_blocks, int q_stride, int out_stride,
                                 float scale, int reach, float softcap, hipStream_t stream) {
    ILM_REQUIRE(n_tiles > 0 && nh > 0 && nkv > 0 && max_blocks > 0, "attn_f32_tile: bad sizes");
    ILM_REQUIRE(nh % nkv == 0, "attn_f32_tile: %d query heads do not divide into %d groups", nh, nkv);
    ILM_REQUIRE(ilm_attn_f32_tile_ok(d, page), "attn_f32_tile: heads of %d, pages of %d keys", d, page);
    ILM_REQUIRE(q_stride % 4 == 0 && out_stride % 4 == 0 && ((uintptr_t)q & 15) == 0 && ((uintptr_t)out & 15) == 0
                    && ((uintptr_t)kc & 15) == 0 && ((uintptr_t)vc & 15) == 0 && (ws == nullptr || ((uintptr_t)ws & 15) == 0),
                "attn_f32_tile: rows must be 16-byte aligned");
    ILM_REQUIRE(ws == nullptr || (nchunks >= 1 && nchunks <= 65535), "attn_f32_tile: %d chunks", nchunks);
    const int G = nh / nkv, nsub = (G + 15) / 16;
    ILM_REQUIRE(n_tiles <= 65535, "attn_f32_tile: %d tiles", n_tiles);
    const int shift = (page & (page - 1)) == 0 ? __builtin_ctz(page) : -1;
    const dim3 grid(nkv * nsub * (G > 8 ? 2 : 1), n_tiles, ws != nullptr ? nchunks : 1);
#define FT_ARGS (float*)out, (float*)ws, (const float*)q, (const float*)kc, (const float*)vc, (const int*)block_tables, (const int*)seg, (const int*)pos, \
                (const int*)tiles, n_tiles, nh, nkv, nsub, page, shift, max_blocks, q_stride, out_stride, scale, reach, softcap
#define FT_RUN(DT_, NW_, TPW_)                                                                                    \
    {                                                                                                             \
        if (ws != nullptr) attn_f32_tile_kernel<DT_, NW_, TPW_, true><<<grid, 64 * NW_, 0, stream>>>(FT_ARGS);    \
        else attn_f32_tile_kernel<DT_, NW_, TPW_, false><<<grid, 64 * NW_, 0, stream>>>(FT_ARGS);                 \
    }
#define FT_CASE(DT_)                    \
    case DT_:                           \
        if (G > 8) FT_RUN(DT_, 4, 1)    \
        else if (G > 4) FT_RUN(DT_, 4, 2) \
        else if (G > 2) FT_RUN(DT_, 2, 4) \
        else FT_RUN(DT_, 1, 8)          \
        break;
    switch (d / 16) {
        FT_CASE(4) FT_CASE(8)
        default: ILM_REQUIRE(false, "attn_f32_tile: head size %d", d);
    }
#undef FT_CASE
#undef FT_ARGS
#undef FT_RUN
    ILM_LAUNCH_CHECK("attn_f32_tile");
    if (ws != nullptr && fold)
        return fa_fold((float*)out, (const float*)ws, (const int*)pos, (const int*)tiles, n_tiles, nullptr, 0, 0, nh, d, nchunks, out_stride, reach, stream);
    return 0;
}
