// whisper_step.hip - the decoder layers of a Whisper step in ONE launch, for as many rows as the compute units have room for.
//
// A step of the launch chain is eight launches a layer, each at its own end: Whisper-tiny's 34 launches of 3 - 10 us are 169 us for weights that stream in 11.  Here blocks stay for all
// layers and hold what they need of the NEXT matrix or head in registers (weight tiles; a head's 384 KB of cached keys and values on eight waves) while others work.  So streaming lies
// beside the chain of dependencies, and what is left of that is eight hand-overs a layer.  These are granules as in lm_step.hip: eight bytes, two bfloat16 values and the tag that says
// whose they are; bounded polls; a request alone on the device.
// A block polls one granule of the values in FRONT of its input, then all of its input: a poll of one granule of the input and then all of it is a round trip more.
//
//  * WS_ALL, small models: a block has ONE task, a few column tiles of one matrix, or the self- or cross-attention of one (row, head).
//  * WS_SHARED, from 1024 columns or several rows on: both attentions of a (row, head) on one block, and tiles of all six matrices on each block that is left, two sets of them in
//    registers at a time - there are not enough compute units to hold a layer's weights and heads.
//
// us a step with the output projection and the sampling (26), chain -> here: 384 columns, 4 layers, one row 167 -> 106, eight 178 -> 128; 768, 12 layers, one 520 -> 300, five 559 -> 378,
// eight 582 -> 415; 1024, 24 layers, one 1070 -> 577, eight 1230 -> 927; 1280, 32 layers, one 1503 -> 920, two 1526 -> 966, eight 1737 -> 1529.  What bounds it: the hand-overs, about
// two us each with the polls, and the short programs between them (a norm 1 - 2, cross-attention 4, products and their sums 1 - 2); eight rows of 1280: 88 blocks for 46 MB of weights, and the
// MLP's 20480 granules in four passes (6 us of a layer's 46; passes of 14 or 20 granules a thread are no faster, two launches a layer with a task a block 55).
//
// Registers: 255 of WS_ALL; WS_SHARED 256, of which 8 spill (20 bytes a lane).
//
// A row has the bits of the launch chain: K is cut and summed as there, and each norm's statistics are dealt and summed as in the kernel that held them (LN_* below).
#include "whisper_step.h"
#include "step_granules.h"

#include <algorithm>
#include <type_traits>

namespace {
// MAX_BLOCKS: a block fills its compute unit's registers; with all 256 units 1280 columns at eight rows take 1474 us a step in place of 1536, but 768 at five 398 for 378, 1024 at one 601 for 577
constexpr int THREADS = 512, WAVES = 8, XPAD = 8, NF = 36, MAX_ROWS = WAVES, D = 64, CJ = 6, SJ = 2, LNG = 5, MAX_BLOCKS = 248;
// attention: a strip of q | k | v a wave, a wave's scores, then probabilities (f32), their halves (bf16), their sums; the waves' partial results
constexpr int LDS_MAX = 160 * 1024;
// WS_SHARED: fragments a wave holds of q | k | v, in whose registers the three square matrices come (two of SH_O, one of SH_CQ), and of the MLP's matrices
constexpr int SH_O = 6, SH_CQ = 5, SH_Q = 2 * SH_O + SH_CQ, SH_F = 24;
constexpr int ATT_SC = 3 * D * 2, ATT_PH = ATT_SC + CJ * 128, ATT_PL = ATT_PH + CJ * 64, ATT_PS = ATT_PL + CJ * 64, ATT_WAVE = ATT_PS + CJ * 16, ATT_LDS = WAVES * (ATT_WAVE + (D + 2) * 4);
// (pointers out of a table in memory: without the address space their loads would be flat ones, which reads of LDS wait for)
template <class T> using Global = const __attribute__((address_space(1))) T*;
template <class T> __device__ __forceinline__ Global<T> global(const T* p) { return (Global<T>)(uintptr_t)p; }
enum { LN_NONE, LN_GLUE, LN_SLICES, LN_WAVE };         // statistics as k_glue4, as k_attn_cross (slices of K a wave), as k_gemm_skinny_norm (a row a wave)
enum { TO_T, TO_RESID, TO_GELU };

struct Exch { unsigned q, at, h1, cq, ca, hb, act, h2, layer; };
__host__ __device__ inline Exch exch_layout(int d, int ff, int rows) {
    Exch e;
    unsigned a = 0;
    e.q = a; a += rows * 3 * d * 4;
    e.at = a; a += rows * d * 4;
    e.h1 = a; a += rows * d * 4;
    e.cq = a; a += rows * d * 4;
    e.ca = a; a += rows * d * 4;
    e.hb = a; a += rows * d * 4;
    e.act = a; a += rows * ff * 4;
    e.h2 = a; a += rows * d * 4;
    e.layer = a;
    return e;
}
// x (rows XPAD columns apart more, so that the rows of a fragment are in different banks) | what the columns without a row read (zeros) and write | partial sums | table of fragments | a norm's weights
struct Lds { int none, part, tab, wb, total; };
__host__ __device__ inline Lds lds_layout(int k_max, int rows, int units) {
    Lds l;
    int a = (k_max + XPAD) * rows * 2;
    l.none = a; a += 128;
    l.part = a; a += units * rows * 64;
    l.tab = a; a += WAVES * NF * 4;
    l.wb = a; a += 2 * 256 * LNG * 2;
    l.total = a > ATT_LDS ? a : ATT_LDS;
    return l;
}
__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ const WsParams& args() { return step_args<WsParams>(); }
// `one`, the same for all lanes of the wave, until it carries `tag`
__device__ __forceinline__ bool await(bool hasty, const unsigned char* one, unsigned tag, int lane) {
    u64 t0 = 0;
    for (int n = 0;; ++n) {
        unsigned v = tag;
        if (lane == 0) v = (unsigned)(__hip_atomic_load(reinterpret_cast<const u64*>(one), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 32);
        if ((unsigned)__builtin_amdgcn_readfirstlane(v) == tag) break;
        if (((n & 63) == 63 || hasty) && !more_time<WsParams>(t0, lane)) return false;
    }
    asm volatile("" ::: "memory");
    return true;
}
// N granules a lane, at(i) granule i's address, until all carry `tag`
template <int N, class At>
__device__ __forceinline__ bool gather(bool hasty, uint32_t (&out)[N], unsigned tag, int lane, At&& at) {
    u64 t0 = 0;
    for (int n = 0;; ++n) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const u64 v = __hip_atomic_load(reinterpret_cast<const u64*>(at(i)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ok = ok && (unsigned)(v >> 32) == tag;
            out[i] = (uint32_t)v;
        }
        if (__all(ok)) break;
        if (((n & 63) == 63 || hasty) && !more_time<WsParams>(t0, lane)) return false;
    }
    asm volatile("" ::: "memory");
    return true;
}

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint2 load2(Global<bf16_t> p) { const u32x2 v = *(Global<u32x2>)p; return make_uint2(v[0], v[1]); }

// ------------------------------------------------------------------------------------------------------------------ a matrix
// A row's norm on one wave, from granules to xs.  `groups` of four columns a lane; the sums of their lanes are added as the chain's kernel added its waves (LN_WAVE: one sum).
template <int KIND> __device__ __forceinline__ int norm_column(int K, int g, int lane) { return KIND == LN_SLICES ? 32 * ((K / 32 * g) / WAVES) + 4 * lane : 4 * (lane + 64 * g); }
template <int KIND> __device__ __forceinline__ int norm_end(int K, int g) { return KIND == LN_SLICES ? 32 * ((K / 32 * (g + 1)) / WAVES) : min(K, 256 * (g + 1)); }
// a norm's weights: asked for together, in front of the wait for its values (column by column behind it they were a round trip each: 1280 columns, 32 layers, two rows 1015 -> 966 us a step), into LDS behind it
struct NormWeights {
    uint2 w[LNG], b[LNG];
    __device__ __forceinline__ void load(int K, Global<bf16_t> pw, Global<bf16_t> pb, int lane) {
#pragma unroll
        for (int g = 0; g < LNG; ++g) {
            const unsigned col = min(4 * (lane + 64 * g), K - 4);
            w[g] = load2(pw + col);
            b[g] = load2(pb + col);
        }
    }
    __device__ __forceinline__ void store(bf16_t* wb, int K, int lane) const {
#pragma unroll
        for (int g = 0; g < LNG; ++g) {
            const int col = 4 * (lane + 64 * g);
            if (col < K) { *reinterpret_cast<uint2*>(wb + col) = w[g]; *reinterpret_cast<uint2*>(wb + K + col) = b[g]; }
        }
    }
};
template <int KIND>
__device__ __forceinline__ bool norm_row(bool hasty, const unsigned char* in, unsigned tag, bf16_t* row, const bf16_t* wb, int K, float eps, int lane) {
    constexpr int G = KIND == LN_SLICES ? WAVES : LNG;
    uint32_t v[2 * G];
    if (!gather<2 * G>(hasty, v, tag, lane, [&](int i) {
            const int col = norm_column<KIND>(K, i >> 1, lane);
            return in + ((unsigned)(col < norm_end<KIND>(K, i >> 1) ? col : K - 4) * 4u + (i & 1) * 8u);
        })) return false;
    float sum[G], sq[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const bool live = norm_column<KIND>(K, g, lane) < norm_end<KIND>(K, g);
        float a = KIND == LN_WAVE && g > 0 ? sum[g - 1] : 0.0f;
        a += live ? bf_lo(v[2 * g]) : 0.0f; a += live ? bf_hi(v[2 * g]) : 0.0f; a += live ? bf_lo(v[2 * g + 1]) : 0.0f; a += live ? bf_hi(v[2 * g + 1]) : 0.0f;
        sum[g] = a;
    }
    auto total = [&](float (&part)[G]) {
        if (KIND == LN_WAVE) return wave_sum_dpp(part[G - 1]);
        float t = 0.0f;
#pragma unroll
        for (int g = 0; g < G; ++g) part[g] = wave_sum_dpp(part[g]);
#pragma unroll
        for (int g = 0; g < G; ++g) t += part[g];
        return t;
    };
    const float mean = total(sum) / (float)K;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const bool live = norm_column<KIND>(K, g, lane) < norm_end<KIND>(K, g);
        const float h[4] = {bf_lo(v[2 * g]), bf_hi(v[2 * g]), bf_lo(v[2 * g + 1]), bf_hi(v[2 * g + 1])};
        float a = KIND == LN_WAVE && g > 0 ? sq[g - 1] : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float dl = h[e] - mean; a += live ? dl * dl : 0.0f; }
        sq[g] = a;
    }
    const float rstd = 1.0f / sqrtf(total(sq) / (float)K + eps);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int col = norm_column<KIND>(K, g, lane);
        if (col < norm_end<KIND>(K, g)) {
            const uint2 w = *reinterpret_cast<const uint2*>(wb + col), b = *reinterpret_cast<const uint2*>(wb + K + col);
            const float h[4] = {bf_lo(v[2 * g]), bf_hi(v[2 * g]), bf_lo(v[2 * g + 1]), bf_hi(v[2 * g + 1])}, wv[4] = {bf_lo(w.x), bf_hi(w.x), bf_lo(w.y), bf_hi(w.y)}, bv[4] = {bf_lo(b.x), bf_hi(b.x), bf_lo(b.y), bf_hi(b.y)};
            bf16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f32_to_bf16(fmaf((h[e] - mean) * rstd, wv[e], bv[e]));
            *reinterpret_cast<uint2*>(row + col) = make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
        }
    }
    return true;
}

// where a matrix's values come from and go to, in a layer's granules
struct Edge { unsigned near, in, out, res; };
// A wave's part of matrix R in a block: the fragments of a few column tiles, at most N, in w[F0 ..) of its registers
template <int R, int LN, int TO, int F0, int N>
struct Task {
    unsigned ent;                                                           // fragment f in lane f (ws_table)
    int n, block;
    __device__ __forceinline__ int tiles(const WsRole& ro) const { return min(ro.per, ro.tiles - block * ro.per); }
    // in the order of ws_table, those of tiles that the last block does not have left out; behind them the last one's weights times zero
    __device__ __forceinline__ void deal(unsigned char* smem, const Lds& l, int blk, int lane, int wave) {
        const WsParams& p = args();
        block = blk;
        unsigned* tab = reinterpret_cast<unsigned*>(smem + l.tab) + wave * NF;
        const unsigned e = lane < NF ? p.table[(R * WAVES + wave) * NF + lane] : 0u;
        const bool have = (e >> 13 & 1u) && (int)(e >> 8 & 15u) < tiles(p.role[R]);
        const u64 all = __ballot(have);
        n = __builtin_amdgcn_readfirstlane((int)__popcll(all));
        if (have) tab[__popcll(all & ((1ull << lane) - 1ull))] = e;
        wave_lds_fence();
        ent = n == 0 ? 0u : lane < n ? tab[lane] : tab[n - 1] & ~(3u << 12);
        wave_lds_fence();
    }
    // fragments [G0, G1) of a layer
    template <int G0 = 0, int G1 = N, int NW>
    __device__ __forceinline__ void request(bf16x8_t (&w)[NW], int li, int lane) const {
        const WsParams& p = args();
        const int KT = p.role[R].KT;
        const Global<bf16x8_t> base = (Global<bf16x8_t>)global(p.layers[li].w[R]) + (size_t)(block * p.role[R].per) * KT * 64 + lane;
#pragma unroll
        for (int g = G0; g < G1; g += 4)
            if (g < n) {
#pragma unroll
                for (int f = g; f < g + 4 && f < G1; ++f) {
                    const unsigned e = __builtin_amdgcn_readlane(ent, f);
                    w[F0 + f] = __builtin_nontemporal_load(base + ((e >> 8 & 15u) * KT + (e & 255u)) * 64);
                }
            }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void weights(NormWeights& nw, int li, int lane, int wave) const {
        if constexpr (LN != LN_NONE) {
            constexpr int which = LN == LN_GLUE ? 0 : LN == LN_SLICES ? 1 : 2;
            const WsParams& p = args();
            if (wave < p.rows) nw.load(p.role[R].KT * 32, global(p.layers[li].lnw[which]), global(p.layers[li].lnb[which]), lane);
        }
    }
    // the input of a layer, from the values at `src`, into xs; false: stop
    __device__ __forceinline__ bool take(unsigned char* smem, const Lds& l, const NormWeights& nw, const unsigned char* src, unsigned tag, int id, int wave) const {
        const WsParams& p = args();
        const int K = p.role[R].KT * 32, KP = K + XPAD, rows = p.rows, lane = id & 63;
        const bool hasty = p.limit == 0;
        bf16_t* xs = reinterpret_cast<bf16_t*>(smem);
        if constexpr (LN != LN_NONE) {
            if (wave >= rows) return true;
            bf16_t* wb = reinterpret_cast<bf16_t*>(smem + l.wb);
            nw.store(wb, K, lane);
            return norm_row<LN>(hasty, src + (size_t)wave * K * 4, tag, xs + wave * KP, wb, K, p.eps, lane);
        }
        const int total = rows * (K / 2);
        auto some = [&](auto count, int b0) {
            constexpr int C = decltype(count)::value;
            if (b0 + wave * 64 >= total) return true;                       // (nothing for this wave)
            uint32_t v[C];
            if (!gather<C>(hasty, v, tag, lane, [&](int i) { return src + (unsigned)min(b0 + id + i * THREADS, total - 1) * 8u; })) return false;
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const int g = b0 + id + i * THREADS;
                if (g < total) reinterpret_cast<uint32_t*>(xs)[g + g / (K / 2) * (XPAD / 2)] = v[i];
            }
            return true;
        };
        int b0 = 0;
        for (; total - b0 > 6 * THREADS; b0 += 10 * THREADS)                // (several rows: a pass is a round trip)
            if (!some(std::integral_constant<int, 10>{}, b0)) return false;
        for (; total - b0 > THREADS; b0 += 3 * THREADS)
            if (!some(std::integral_constant<int, 3>{}, b0)) return false;
        return b0 >= total || some(std::integral_constant<int, 1>{}, b0);
    }
    // a layer: input, products, sums, values.  false: stop
    template <int NW>
    __device__ __forceinline__ bool layer(unsigned char* smem, const Lds& l, bf16x8_t (&w)[NW], int layer, int tid, int wave, const Edge& at, unsigned exch_layer, unsigned tag) const {
        int li = layer, id = tid;
        asm volatile("" : "+s"(li), "+v"(id));                             // (addresses kept over all layers are registers that the weights need)
        const WsParams& p = args();
        const WsRole ro = p.role[R];
        const int lane = tid & 63, K = ro.KT * 32, KP = K + XPAD, P = ro.S * ro.ksb, tile0 = block * ro.per, nt = tiles(ro), cols = ro.tiles * 16, rows = p.rows;
        const bool hasty = p.limit == 0;
        float* part = reinterpret_cast<float*>(smem + l.part);
        // the values that a thread sums: columns 2 c2, 2 c2 + 1 of tile t, row m
        const int pairs = nt * 8, m = id / pairs, rest = id - m * pairs, t = rest >> 3, col = (tile0 + t) * 16 + (rest & 7) * 2;
        const bool mine = id < pairs * rows;
        unsigned char* now = p.exch + (size_t)exch_layer * li;
        // what the values in front of the input say is near, and what is there before it: bias, the norm's weights
        unsigned char* const src = R == WS_QKV ? now - exch_layer : now;
        NormWeights nw;
        if (R != WS_QKV || li > 0) weights(nw, li, lane, wave);
        if ((R != WS_QKV || li > 0) && at.near != at.in && (LN == LN_NONE || wave < rows) && !await(hasty, src + at.near, tag, lane)) return false;
        const uint32_t bias = mine && p.layers[li].b[R] ? *(Global<uint32_t>)global(p.layers[li].b[R] + col) : 0u;
        if ((R != WS_QKV || li > 0) && !take(smem, l, nw, src + at.in, tag, id, wave)) return false;
        // the residual: there where the input, which is made of it, has come (its tag is looked at behind the products all the same)
        const unsigned char* from = (R == WS_O ? now - exch_layer : now) + at.res + ((size_t)m * cols + col) * 4;
        u64 res = (u64)tag << 32;
        if (TO == TO_RESID && mine) {
            if (R == WS_O && li == 0) res |= *reinterpret_cast<const uint32_t*>(p.h0 + (size_t)m * p.d + col);
            else res = __hip_atomic_load(reinterpret_cast<const u64*>(from), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        bar();
        {
            const int xr = lane & 15, kg = lane >> 4;
            const bool row = xr < rows;
            const unsigned xstep = row ? 64 : 0, xbase = row ? xr * KP * 2 + kg * 16 : l.none, ustep = row ? rows * 64 : 0, ubase = row ? l.part + xr * 64 + kg * 16 : l.none + 64 + kg * 16;
            f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < N; g += 4)
                if (g < n) {
                    bf16x8_t x[4];
#pragma unroll
                    for (int f = 0; f < 4 && g + f < N; ++f)
                        x[f] = *reinterpret_cast<const bf16x8_t*>(smem + xbase + __umul24(__builtin_amdgcn_readlane(ent, g + f) & 255u, xstep));
#pragma unroll
                    for (int f = 0; f < 4 && g + f < N; ++f) {
                        const unsigned e = __builtin_amdgcn_readlane(ent, g + f);
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[F0 + g + f], x[f], acc, 0, 0, 0);
                        if (e & (1u << 12)) {
                            *reinterpret_cast<f32x4_t*>(smem + ubase + __umul24(e >> 16, ustep)) = acc;
                            acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                        }
                    }
                }
        }
        bar();
        uint32_t hres = (uint32_t)res;
        if (TO == TO_RESID && !__all((unsigned)(res >> 32) == tag)) {
            bool good = true;
            if (mine && (R != WS_O || li > 0)) {
                uint32_t v[1];
                good = gather<1>(hasty, v, tag, lane, [&](int) { return from; });
                hres = v[0];
            }
            if (!__all(good)) return false;
        }
        if (mine) {
            constexpr int KSB = R == WS_CQ || R == WS_FC1 ? 8 : 4, G = 16 / KSB;
            float a0 = 0.f, a1 = 0.f;
            const float* q = part + (t * P * rows + m) * 16 + (rest & 7) * 2;
            for (int s0 = 0; s0 < ro.S; s0 += G) {
                float2 v[G][KSB];
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int i = 0; i < KSB; ++i) v[g][i] = *reinterpret_cast<const float2*>(q + (min(s0 + g, ro.S - 1) * KSB + i) * rows * 16);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    float b0 = v[g][0].x, b1 = v[g][0].y;
#pragma unroll
                    for (int i = 1; i < KSB; ++i) { b0 += v[g][i].x; b1 += v[g][i].y; }
                    if (s0 + g == 0) { b0 += bf_lo(bias); b1 += bf_hi(bias); }
                    if (s0 + g < ro.S) { a0 += b0; a1 += b1; }
                }
            }
            if (TO == TO_RESID) { a0 = bf_lo(hres) + bf16_round_f32(a0); a1 = bf_hi(hres) + bf16_round_f32(a1); }
            if (TO == TO_GELU) { a0 = gelu_erf(bf16_round_f32(a0)); a1 = gelu_erf(bf16_round_f32(a1)); }
            granule(now + at.out + ((size_t)m * cols + col) * 4, (uint32_t)f32_to_bf16(a0) | (uint32_t)f32_to_bf16(a1) << 16, tag);
        }
        bar();                                                             // (the next weights are asked for behind the stores)
        return true;
    }
};
// the rows in front of the first layer into xs
__device__ __forceinline__ void first_rows(unsigned char* smem, int tid) {
    const WsParams& p = args();
    for (int i = tid; i < p.rows * (p.d / 8); i += THREADS) {
        const int r = i / (p.d / 8), k = (i - r * (p.d / 8)) * 8;
        *reinterpret_cast<uint4*>(smem + 2 * (r * (p.d + XPAD) + k)) = *reinterpret_cast<const uint4*>(p.x0 + xpk_index(r, k, 1));
    }
}
// behind the last layer: the decoder's norm
template <class T>
__device__ __forceinline__ void last_rows(const T& qkv, unsigned char* smem, const Lds& l, int tid, int wave, const Edge& at, unsigned exch_layer, unsigned tag) {
    const WsParams& p = args();
    const unsigned char* src = p.exch + (size_t)exch_layer * (p.L - 1);
    NormWeights nw;
    qkv.weights(nw, p.L, tid & 63, wave);
    if ((wave < p.rows && !await(p.limit == 0, src + at.near, tag, tid & 63)) || !qkv.take(smem, l, nw, src + at.in, tag, tid, wave)) return;
    bar();
    for (int i = tid; i < p.rows * (p.d / 8); i += THREADS) {
        const int r = i / (p.d / 8), k = (i - r * (p.d / 8)) * 8;
        *reinterpret_cast<uint4*>(args().x_out + xpk_index(r, k, 1)) = *reinterpret_cast<const uint4*>(smem + 2 * (r * (p.d + XPAD) + k));
    }
}
__device__ __forceinline__ void clear_lds(unsigned char* smem, const Lds& l, int tid) {
    if (tid < 32) reinterpret_cast<unsigned*>(smem + l.none)[tid] = 0;
    const int n = args().units * args().rows * 16;
    for (int i = tid; i < n; i += THREADS) reinterpret_cast<float*>(smem + l.part)[i] = 0.f;          // (a piece without a K-tile stays zero)
}

// one matrix a block (WS_ALL)
template <int R, int LN, int TO>
__device__ __forceinline__ void matrix(unsigned char* smem, int block, int tid, const Edge at, unsigned exch_layer, unsigned tag) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), L = args().L;
    const Lds l = lds_layout(args().k_max, args().rows, args().units);
    clear_lds(smem, l, tid);
    bf16x8_t w[NF];
    Task<R, LN, TO, 0, NF> t;
    t.deal(smem, l, block, lane, wave);
    t.request(w, 0, lane);
    if (R == WS_QKV) first_rows(smem, tid);
    for (int li = 0; li < L; ++li) {
        if (!t.layer(smem, l, w, li, tid, wave, at, exch_layer, tag)) return;
        if (li + 1 < L) t.request(w, li + 1, lane);
    }
    if (R == WS_QKV && block == 0) last_rows(t, smem, l, tid, wave, at, exch_layer, tag);
}

// Column tiles of every matrix a block (WS_SHARED).  Its registers hold two of four sets at a time: q | k | v or the three square matrices; either of the MLP.
// A set is asked for as soon as the one whose registers it takes has been multiplied.
__device__ __forceinline__ void matrices(unsigned char* smem, int block, int tid, const Exch& ex, unsigned tag) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), L = args().L, blocks = args().self_first;
    const Lds l = lds_layout(args().k_max, args().rows, args().units);
    clear_lds(smem, l, tid);
    bf16x8_t w[SH_Q + SH_F];
    Task<WS_QKV, LN_GLUE, TO_T, 0, SH_Q> qkv;
    Task<WS_O, LN_NONE, TO_RESID, 0, SH_O> o;
    Task<WS_CQ, LN_SLICES, TO_T, SH_O, SH_CQ> cq;
    Task<WS_CO, LN_NONE, TO_RESID, SH_O + SH_CQ, SH_O> co;
    Task<WS_FC1, LN_WAVE, TO_GELU, SH_Q, SH_F> fc1;
    Task<WS_FC2, LN_NONE, TO_RESID, SH_Q, SH_F> fc2;
    auto place = [&](auto& t, int role) {
        const int b = block - args().role[role].first;
        t.deal(smem, l, b < 0 ? b + blocks : b, lane, wave);
        return t.block < args().role[role].blocks;
    };
    const bool hq = place(qkv, WS_QKV), ho = place(o, WS_O), hcq = place(cq, WS_CQ), hco = place(co, WS_CO), h1 = place(fc1, WS_FC1), h2 = place(fc2, WS_FC2);
    const Edge eq{ex.act, ex.h2, ex.q, 0}, eo{ex.q, ex.at, ex.h1, ex.h2}, ecq{ex.at, ex.h1, ex.cq, 0}, eco{ex.cq, ex.ca, ex.hb, ex.h1}, e1{ex.ca, ex.hb, ex.act, 0}, e2{ex.act, ex.act, ex.h2, ex.hb};
    if (hq) qkv.request(w, 0, lane);
    first_rows(smem, tid);
    for (int li = 0; li < L; ++li) {
        if (hq && !qkv.layer(smem, l, w, li, tid, wave, eq, ex.layer, tag)) return;
        if (ho) o.request(w, li, lane);
        if (hcq) cq.request(w, li, lane);
        if (hco) co.request(w, li, lane);
        if (ho && !o.layer(smem, l, w, li, tid, wave, eo, ex.layer, tag)) return;
        if (hcq && !cq.layer(smem, l, w, li, tid, wave, ecq, ex.layer, tag)) return;
        if (h1) fc1.request(w, li, lane);
        if (hq && li + 1 < L) qkv.request<0, SH_O + SH_CQ>(w, li + 1, lane);
        if (hco && !co.layer(smem, l, w, li, tid, wave, eco, ex.layer, tag)) return;
        if (hq && li + 1 < L) qkv.request<SH_O + SH_CQ, SH_Q>(w, li + 1, lane);
        if (h1 && !fc1.layer(smem, l, w, li, tid, wave, e1, ex.layer, tag)) return;
        if (h2) fc2.request(w, li, lane);
        if (h2 && !fc2.layer(smem, l, w, li, tid, wave, e2, ex.layer, tag)) return;
    }
    if (block == 0) last_rows(qkv, smem, l, tid, wave, eq, ex.layer, tag);
}

// ------------------------------------------------------------------------------------------------------------------ attention of a (row, head)
// Eight waves, tiles wave, wave + 8, .. of 32 keys each (k_attn_decode's); NJ tiles a wave at most, all in registers before the query is there.  The products, the running maximum over the
// tiles and the order of the sums are k_attn_cross's.
template <int NJ> struct Tiles { bf16x8_t ka[NJ][2][2], va[NJ][4]; };
// what an attention knows of its (row, head) for all layers
template <bool SELF>
struct Head {
    int lane, wave, b, h, pos, kv_len, n_tiles;
    bool live;
    size_t head;
    __device__ __forceinline__ Head(int item, int tid) {
        const WsParams& p = args();
        lane = tid & 63; wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        b = item / p.H; h = item - b * p.H;
        pos = SELF ? p.pos[b] : 0;
        live = p.active[b] != 0;
        kv_len = SELF ? pos + 1 : p.cross_len;
        n_tiles = (kv_len + 31) >> 5;
        head = ((size_t)b * p.H + h) * (SELF ? p.Smax : p.Spad) * D;
    }
    // tiles [J0, J1) of this wave's
    template <int NJ, int J0, int J1>
    __device__ __forceinline__ void load(Tiles<NJ>& t, int li) const {
        const WsParams& p = args();
        const bf16x8_t* kb = reinterpret_cast<const bf16x8_t*>((SELF ? p.self_k + p.self_layer * li : p.cross_k + p.cross_layer * li) + head) + lane;
        const bf16x8_t* vb = reinterpret_cast<const bf16x8_t*>((SELF ? p.self_v + p.self_layer * li : p.cross_v + p.cross_layer * li) + head) + lane;
#pragma unroll
        for (int j = J0; j < J1; ++j) {
            const int tile = min(wave + j * WAVES, n_tiles - 1);              // (a wave with fewer tiles: one that it does not use)
#pragma unroll
            for (int c = 0; c < 4; ++c) t.ka[j][c >> 1][c & 1] = __builtin_nontemporal_load(kb + ((size_t)tile * 4 + c) * 64);
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) t.va[j][dt] = __builtin_nontemporal_load(vb + ((size_t)tile * 4 + dt) * 64);
        }
        asm volatile("" ::: "memory");
    }
};
// One layer.  false: stop
template <int NJ, bool SELF>
__device__ __forceinline__ bool attend(unsigned char* smem, const Head<SELF>& hd, Tiles<NJ>& t, int li, bool hasty, unsigned near_at, unsigned q_at, unsigned out_at, unsigned exch_layer, unsigned tag) {
    const int lane = hd.lane, wave = hd.wave, g4 = lane >> 4, d0 = lane & 15, b = hd.b, h = hd.h, pos = hd.pos, kv_len = hd.kv_len, n_tiles = hd.n_tiles;
    const bool live = hd.live;
    const size_t head = hd.head;
    auto& ka = t.ka;
    auto& va = t.va;
    const WsParams& p = args();
    const int d = p.d;
    const float scale = p.scale;
    unsigned char* own = smem + wave * ATT_WAVE;
    bf16_t* strip = reinterpret_cast<bf16_t*>(own);
    float *sc = reinterpret_cast<float*>(own + ATT_SC), *ps = reinterpret_cast<float*>(own + ATT_PS);
    bf16_t *ph = reinterpret_cast<bf16_t*>(own + ATT_PH), *pl = reinterpret_cast<bf16_t*>(own + ATT_PL);
    float* part = reinterpret_cast<float*>(smem + WAVES * ATT_WAVE);        // [WAVES][D + 2]
    unsigned char* now = p.exch + (size_t)exch_layer * li;
    constexpr int NG = SELF ? 2 : 1;
    uint32_t v[NG];
    if ((!SELF || li > 0) && !await(hasty, now - (SELF ? exch_layer : 0u) + near_at, tag, lane)) return false;
    const unsigned char* from = now + q_at + (size_t)b * (SELF ? 3 : 1) * d * 4 + h * D * 4;
    // q | k | v of the head, 32 granules each; the cross-attention: q
    if (!gather<NG>(hasty, v, tag, lane, [&](int i) {
            const int g = min(lane + 64 * i, SELF ? 95 : 31);
            return from + (size_t)(g >> 5) * d * 4 + (g & 31) * 8;
        })) return false;
#pragma unroll
    for (int i = 0; i < NG; ++i)
        if (lane + 64 * i < (SELF ? 96 : 32)) reinterpret_cast<uint32_t*>(strip)[lane + 64 * i] = v[i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    bf16x8_t qf[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) qf[c] = *reinterpret_cast<const bf16x8_t*>(strip + c * 32 + g4 * 8);
    if (SELF && live) {
        // the new key, in the registers of the wave whose tile it is and in the cache
        const int tile = pos >> 5, pr = pos & 31, prow = ((pr >> 3) << 2) | (pr & 3), half = (pr >> 2) & 1;
        if ((tile & (WAVES - 1)) == wave) {
            const int jn = tile / WAVES;
            bf16x8_t* kc = reinterpret_cast<bf16x8_t*>(p.self_k + p.self_layer * li + head) + ((size_t)tile * 2 + half) * 2 * 64 + lane;
            bf16_t* vc = p.self_v + p.self_layer * li + head;
            if (d0 == prow) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const bf16x8_t kn = *reinterpret_cast<const bf16x8_t*>(strip + D + c * 32 + g4 * 8);
                    kc[c * 64] = kn;
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        if (j == jn) { if (half) ka[j][1][c] = kn; else ka[j][0][c] = kn; }
                }
            }
            if (g4 == (pr >> 3)) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) {
                    const bf16_t vn = strip[2 * D + dt * 16 + d0];
                    vc[(((size_t)tile * 4 + dt) * 64 + lane) * 8 + (pr & 7)] = vn;
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if (j == jn && e == (pr & 7)) va[j][dt][e] = (short)vn;
                }
            }
        }
    }
    // Scores stand in all sixteen columns: through LDS a lane gets one key of every second tile, and gives the probabilities back (sixteen times the vector work otherwise:
    // 4.9 us at six tiles a wave)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        f32x4_t S0 = (f32x4_t){0.f, 0.f, 0.f, 0.f}, S1 = S0;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            S0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[j][0][c], qf[c], S0, 0, 0, 0);
            S1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[j][1][c], qf[c], S1, 0, 0, 0);
        }
        if (d0 == 0) { *reinterpret_cast<f32x4_t*>(sc + j * 32 + g4 * 8) = S0; *reinterpret_cast<f32x4_t*>(sc + j * 32 + g4 * 8 + 4) = S1; }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (LDS operations of one wave execute in order)
    float m_run = -INFINITY, l_run = 0.0f, alpha[NJ], x[NJ / 2], mx[NJ / 2];
    const int up = lane >> 5;
#pragma unroll
    for (int i = 0; i < NJ / 2; ++i) {
        const float v = sc[i * 64 + lane] * scale;
        x[i] = (wave + (2 * i + up) * WAVES) * 32 + (lane & 31) < kv_len ? v : -INFINITY;
        mx[i] = x[i];
    }
#pragma unroll
    for (int k = 1; k < 32; k <<= 1)
#pragma unroll
        for (int i = 0; i < NJ / 2; ++i) mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], k, 64));
#pragma unroll
    for (int i = 0; i < NJ / 2; ++i) {
        const float m0 = fmaxf(m_run, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[i]), 0)));
        alpha[2 * i] = __expf(m_run - m0);
        const bool two = wave + (2 * i + 1) * WAVES < n_tiles;         // (a group of five)
        const float m1 = two ? fmaxf(m0, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[i]), 32))) : m0;
        alpha[2 * i + 1] = __expf(m0 - m1);
        m_run = wave + 2 * i * WAVES < n_tiles ? m1 : m_run;
        const float pe = __expf(x[i] - (up ? m1 : m0));
        const bf16_t hb = f32_to_bf16(pe);
        sc[i * 64 + lane] = pe;
        ph[i * 64 + lane] = hb;
        pl[i * 64 + lane] = f32_to_bf16(pe - bf16_to_f32(hb));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane < NJ * 4) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(sc + lane * 8), c = *reinterpret_cast<const f32x4_t*>(sc + lane * 8 + 4);
        float psum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) psum += e < 4 ? a[e & 3] : c[e & 3];
        ps[lane] = psum;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    f32x4_t O[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) O[dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (wave + j * WAVES < n_tiles) {
            l_run = l_run * alpha[j] + ps[j * 4 + g4];
            const bf16x8_t fh = *reinterpret_cast<const bf16x8_t*>(ph + j * 32 + g4 * 8), fl = *reinterpret_cast<const bf16x8_t*>(pl + j * 32 + g4 * 8);   // P in bf16 hi + lo parts
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                f32x4_t o = O[dt];
                o[0] *= alpha[j];                                       // (row 0 of O is read, the others are copies without their factors)
                o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh, va[j][dt], o, 0, 0, 0);
                O[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl, va[j][dt], o, 0, 0, 0);
            }
        }
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    if (g4 == 0) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) part[wave * (D + 2) + dt * 16 + d0] = O[dt][0];
        if (d0 < 2) part[wave * (D + 2) + D + d0] = d0 ? l_run : m_run;
    }
    bar();
    if (wave == 0) {
        float M = -INFINITY, num = 0.0f, den = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) M = fmaxf(M, part[w * (D + 2) + D]);
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float f = __expf(part[w * (D + 2) + D] - M);
            num += f * part[w * (D + 2) + lane];
            den += f * part[w * (D + 2) + D + 1];
        }
        const uint32_t o = live ? f32_to_bf16(num / den) : 0u, next = __shfl_xor(o, 1, 64);
        if (!(lane & 1)) granule(now + out_at + ((size_t)b * d + h * D + lane) * 4, o | next << 16, tag);
    }
    bar();
    return true;
}
template <int NJ, bool SELF>
__device__ __forceinline__ void attention(unsigned char* smem, int item, int tid, unsigned near_at, unsigned q_at, unsigned out_at, unsigned exch_layer, unsigned tag) {
    const bool hasty = args().limit == 0;
    const int L = args().L;
    const Head<SELF> hd(item, tid);
    Tiles<NJ> t;
    hd.template load<NJ, 0, NJ>(t, 0);
    for (int li = 0; li < L; ++li) {
        if (!attend<NJ, SELF>(smem, hd, t, li, hasty, near_at, q_at, out_at, exch_layer, tag)) return;
        if (li + 1 < L) hd.template load<NJ, 0, NJ>(t, li + 1);
    }
}
// Both attentions of a (row, head) (WS_SHARED).  The cross-attention's tiles are asked for behind the layer before, but those whose registers hold the self-attention's.
__device__ __forceinline__ void attentions(unsigned char* smem, int item, int tid, const Exch& ex, unsigned tag) {
    const bool hasty = args().limit == 0;
    const int L = args().L;
    const Head<true> own(item, tid);
    const Head<false> cross(item, tid);
    constexpr int EARLY = CJ - SJ;
    for (int li = 0; li < L; ++li) {
        Tiles<SJ> t;
        Tiles<CJ> x;
        own.template load<SJ, 0, SJ>(t, li);
        cross.template load<CJ, 0, EARLY>(x, li);
        if (!attend<SJ, true>(smem, own, t, li, hasty, ex.h2, ex.q, ex.at, ex.layer, tag)) return;
        cross.template load<CJ, EARLY, CJ>(x, li);
        if (!attend<CJ, false>(smem, cross, x, li, hasty, ex.h1, ex.cq, ex.ca, ex.layer, tag)) return;
    }
}

template <int WHAT>
__global__ void __launch_bounds__(THREADS, 2) k_whisper_step(WsParams) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int blk = blockIdx.x, tid = threadIdx.x;
    const Exch ex = exch_layout(args().d, args().ff, args().rows);
    const unsigned tag = args().sync[SYNC_TAG] + 1;
    if constexpr (WHAT == WS_SHARED) {
        if (blk >= args().self_first) attentions(smem, blk - args().self_first, tid, ex, tag);
        else matrices(smem, blk, tid, ex, tag);
    } else if (blk >= args().cross_first) attention<CJ, false>(smem, blk - args().cross_first, tid, ex.h1, ex.cq, ex.ca, ex.layer, tag);
    else if (blk >= args().self_first) attention<SJ, true>(smem, blk - args().self_first, tid, ex.h2, ex.q, ex.at, ex.layer, tag);
    else if (blk >= args().role[WS_FC2].first) matrix<WS_FC2, LN_NONE, TO_RESID>(smem, blk - args().role[WS_FC2].first, tid, {ex.hb, ex.act, ex.h2, ex.hb}, ex.layer, tag);
    else if (blk >= args().role[WS_FC1].first) matrix<WS_FC1, LN_WAVE, TO_GELU>(smem, blk - args().role[WS_FC1].first, tid, {ex.ca, ex.hb, ex.act, 0}, ex.layer, tag);
    else if (blk >= args().role[WS_CO].first) matrix<WS_CO, LN_NONE, TO_RESID>(smem, blk - args().role[WS_CO].first, tid, {ex.cq, ex.ca, ex.hb, ex.h1}, ex.layer, tag);
    else if (blk >= args().role[WS_CQ].first) matrix<WS_CQ, LN_SLICES, TO_T>(smem, blk - args().role[WS_CQ].first, tid, {ex.at, ex.h1, ex.cq, 0}, ex.layer, tag);
    else if (blk >= args().role[WS_O].first) matrix<WS_O, LN_NONE, TO_RESID>(smem, blk - args().role[WS_O].first, tid, {ex.q, ex.at, ex.h1, ex.h2}, ex.layer, tag);
    else matrix<WS_QKV, LN_GLUE, TO_T>(smem, blk, tid, {ex.act, ex.h2, ex.q, 0}, ex.layer, tag);
    if (blk == 0 && tid == 0) {
        const WsParams& p = args();                               // (the block that ends last: it waits for the others' values)
        p.sync[SYNC_TAG] = tag;
    }
}
// Pieces to waves, the longest first, each to the wave with the least: fragments of the fullest wave; out: WAVES x NF entries of
// K-tile | tile << 8 | last of its piece << 12 | 1 << 13 | piece << 16 (0: none)
int ws_table(const WsRole& r, int per, unsigned* out) {
    struct Piece { int unit, tile, k0, k1; };
    std::vector<Piece> v;
    const int P = r.S * r.ksb;
    for (int u = 0; u < per * P; ++u) {
        const int pc = u % P, ks = pc / r.ksb, w = pc % r.ksb, a = r.KT * ks / r.S, len = r.KT * (ks + 1) / r.S - a;
        v.push_back({u, u / P, a + len * w / r.ksb, a + len * (w + 1) / r.ksb});
    }
    std::stable_sort(v.begin(), v.end(), [](const Piece& a, const Piece& b) { return a.k1 - a.k0 > b.k1 - b.k0; });
    int n[WAVES] = {};
    for (const Piece& c : v) {
        const int w = (int)(std::min_element(n, n + WAVES) - n);
        for (int k = c.k0; k < c.k1; ++k, ++n[w])
            if (out && n[w] < NF) out[w * NF + n[w]] = (unsigned)k | (unsigned)c.tile << 8 | (k + 1 == c.k1 ? 1u << 12 : 0u) | 1u << 13 | (unsigned)c.unit << 16;
    }
    return *std::max_element(n, n + WAVES);
}
int lds_bytes(const WsParams& p) { return lds_layout(p.k_max, p.rows, p.units).total; }
bool fits(WsParams& p) {
    p.units = 0;
    for (const WsRole& r : p.role) {
        p.units = std::max(p.units, r.per * r.S * r.ksb);
        if (r.per > 8 || r.per * 8 * p.rows > THREADS) return false;
    }
    return lds_bytes(p) <= LDS_MAX;
}
// a matrix a block, an attention a block; false: more than there are compute units
bool plan_all(WsParams& p, int cus) {
    p.what = WS_ALL;
    for (WsRole& r : p.role) r.per = 1;
    for (;;) {                                                              // more tiles a block, where that makes the shortest block, until a compute unit has one block
        int total = 2 * p.rows * p.H, best = -1, cost = 0;
        for (int i = 0; i < WS_ROLES; ++i) {
            WsRole& r = p.role[i];
            r.blocks = (r.tiles + r.per - 1) / r.per;
            total += r.blocks;
            const int f = r.blocks > 1 ? ws_table(r, r.per + 1, nullptr) : NF + 1;
            if (r.per < 8 && f <= NF && (best < 0 || f < cost)) { best = i; cost = f; }
        }
        if (total <= std::min(cus, MAX_BLOCKS)) break;
        if (best < 0) return false;
        ++p.role[best].per;
    }
    int at = 0;
    for (WsRole& r : p.role) { r.first = at; at += r.blocks; }
    p.self_first = at; at += p.rows * p.H;
    p.cross_first = at; at += p.rows * p.H;
    p.blocks = at;
    return fits(p);
}
int fullest(const WsParams& p) {
    int n = 0;
    for (const WsRole& r : p.role) n = std::max(n, ws_table(r, r.per, nullptr));
    return n;
}
// every matrix on the blocks that the attentions leave, both attentions of a (row, head) on one
bool plan_shared(WsParams& p, int cus) {
    p.what = WS_SHARED;
    int most = 0, blocks = std::min(cus, MAX_BLOCKS) - p.rows * p.H, at = 0;
    for (const WsRole& r : p.role) {
        most = std::max(most, r.tiles);
        if (r.KT / r.S < r.ksb) return false;                              // (a piece without a K-tile)
    }
    blocks = std::min(blocks, most);
    if (blocks < 1) return false;
    const int room[WS_ROLES] = {SH_Q, SH_O, SH_CQ, SH_O, SH_F, SH_F};
    for (int i = 0; i < WS_ROLES; ++i) {
        WsRole& r = p.role[i];
        r.per = (r.tiles + blocks - 1) / blocks;
        r.blocks = (r.tiles + r.per - 1) / r.per;
        r.first = at;                                                       // (matrices of fewer tiles than blocks beside each other)
        at = (at + r.blocks) % blocks;
        if (r.per > 8 || ws_table(r, r.per, nullptr) > room[i]) return false;
    }
    p.self_first = blocks;
    p.cross_first = p.blocks = blocks + p.rows * p.H;
    return fits(p);
}
}

size_t ws_exch_bytes(const WsParams& p) { return (size_t)exch_layout(p.d, p.ff, p.rows).layer * p.L; }

bool ws_plan(WsParams& p, int device) {
    if (p.rows < 1 || p.rows > MAX_ROWS || p.L < 1 || p.d % 64 || p.d > 256 * LNG || p.d != p.H * D || p.ff % 32 || p.Smax > 32 * WAVES * SJ || p.Smax % 32 ||
        p.cross_len > 32 * WAVES * CJ || p.cross_len <= 32 * WAVES * (CJ - 1) || p.Spad < (p.cross_len + 31) / 32 * 32) return false;
    p.k_max = 0;
    for (const WsRole& r : p.role) {
        if (r.KT > 255 || r.S < 1 || r.S > 8 || ws_table(r, 1, nullptr) > NF) return false;
        p.k_max = std::max(p.k_max, r.KT * 32);
    }
    int cus = 0, lds = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device) != hipSuccess || lds < LDS_MAX) return false;
    for (auto f : {reinterpret_cast<const void*>(&k_whisper_step<WS_ALL>), reinterpret_cast<const void*>(&k_whisper_step<WS_SHARED>)})
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX) != hipSuccess) { (void)hipGetLastError(); return false; }
    // One matrix a block while its blocks hold few fragments; from there on their sums and the few compute units a matrix has cost more than what blocks of all matrices wait for
    // (us a step, one / all a block: 768 columns, 12 layers, four rows - 15 fragments - 360 / 364, five 409 / 378; 1024, 24 layers, one row - 20 - 608 / 583; 1280, 32 layers, one 995 / 931)
    if (plan_all(p, cus) && fullest(p) <= 16) return true;
    return plan_shared(p, cus) || plan_all(p, cus);
}

std::vector<unsigned> ws_tables(const WsParams& p) {
    std::vector<unsigned> t(WS_ROLES * WAVES * NF, 0u);
    for (int i = 0; i < WS_ROLES; ++i) ws_table(p.role[i], p.role[i].per, t.data() + i * WAVES * NF);
    return t;
}

void launch_whisper_step(const WsParams& p, hipStream_t s) {
    if (p.what == WS_SHARED) hipLaunchKernelGGL(k_whisper_step<WS_SHARED>, dim3(p.blocks), dim3(THREADS), lds_bytes(p), s, p);
    else hipLaunchKernelGGL(k_whisper_step<WS_ALL>, dim3(p.blocks), dim3(THREADS), lds_bytes(p), s, p);
}
