// lm_step.hip - the layers of a decode step of one or two rows in ONE launch.
//
// A launch chain pays every layer's five kernels their ramp and tail: at one row of the 3B model 50 us a layer for 201 MB of weights that stream in 31.  Here 256 blocks, one a compute
// unit, stay for all layers; a block owns the same column tiles of each matrix in every layer, its weights are asked for ahead of the values they are multiplied with, and what is left
// of a hand-over is the way of a few kilobytes from compute unit to compute unit.  28 layers of 3072 / 8192, one row, contexts to 110: 50.7 -> 43.8 us a layer (4.6 TB/s); two rows 53.7 -> 49.2.
//
//  * Twelve waves a block.  Eight MATRIX waves multiply: the K ranges (`pieces`) of the block's column tiles are dealt to them, a piece being what one wave of the chain takes, in the
//    same order.  The four VECTOR waves do the rest: they add the pieces as the chain adds its waves and slabs, round where it rounds, and do residual, RMSNorm and attention with
//    the chain's threads, tiles and sums.  So a row has the bits of the launch chain, alone or in a larger batch.
//  * Weights go to LDS without registers between (16 bytes a lane, four kilobytes a group), through a ring of each matrix wave; its oldest groups move on into registers while it has
//    nothing to multiply: 28 KB a wave, 224 KB a compute unit ahead.  In that time a wave keeps three kilobytes under way (FLIGHT): requests that wait in a compute unit's
//    queue stand in front of the vector waves' stores and polls (us a layer at one row with 1, 2, 3, 4, 8: 49.7, 44.0, 43.8, 44.5, 45.7), and none is made between a phase's sums and
//    the stores of its values (45.9 without that).
//  * A hand-over between blocks is a GRANULE, eight bytes: two bfloat16 values and the tag (launch and layer) that says whose they are, one agent-scope store, polled by whoever needs
//    it.  Nothing is waited for behind the store and there is no flag (with lines of values, a flag behind their acknowledgement and a gather: 59 us).  A wave polls one granule until
//    it is there, then all of its own: every block polling all of a vector is as much traffic as the weights (46.3 against 47.5).  Every layer has granules of its own, so none is
//    overwritten in a launch that reads it; tags grow over the launches of a request and the granules are cleared in front of it.
//  * Registers: 168 for each of twelve waves, of which 37 spill (112 bytes a lane).
//  * Polls end: out of time (StepParams::limit: another stream holds compute units), a block raises `fail`, which all others see, every wave leaves, and the request runs again on the launch
//    chain.  Two launches that each hold part of the compute units would wait for each other: a request takes this path while its call is alone on the device (DeviceTurn, common.h).
#include "step_granules.h"

#include <stdio.h>

namespace {
constexpr int CU = 256, MWAVES = 8, VWAVES = 4, THREADS = (MWAVES + VWAVES) * 64, VT = VWAVES * 64, MAX_ROWS = 2, TAB = 16, VIRT = 8, CPT = 3;
constexpr int AHEAD = 3, FLIGHT = 3;

// per layer: q|k|v, attention, h behind it, h behind the layer, activation: granules [row][columns / 2] of {two values, tag}
struct Layout { unsigned q, a, h1, act, h2, layer; };
__host__ __device__ inline Layout exch_layout(int d, int ff, int H, int Hkv, int D, int rows) {
    Layout l;
    unsigned at = 0;
    l.q = at; at += rows * (H + 2 * Hkv) * D * 4;
    l.a = at; at += rows * H * D * 4;
    l.h1 = at; at += rows * d * 4;
    l.h2 = at; at += rows * d * 4;
    l.act = at; at += rows * ff * 4;
    l.layer = at;
    return l;
}
struct Lds { int ring, xs, strip, so, sm, part, tab, red, misc, total; };
__host__ __device__ inline Lds lds_layout(int ring, int k_max, int rows, int G, int max_units) {
    Lds l;
    int at = 0;
    l.ring = at; at += MWAVES * ring * 1024;
    l.xs = at;                                                             // the attention's areas lie over the operand: one is read when the other is not
    l.strip = at; l.so = at + VWAVES * (G + 3) * 128 * 4; l.sm = l.so + VIRT * G * 128 * 4;
    const int attn = l.sm + 2 * VIRT * 16 * 4 - at, xs = k_max / 32 * 64 * rows;
    at += attn > xs ? attn : xs;
    l.part = at; at += max_units * rows * 64;
    l.tab = at; at += MWAVES * TAB * 8;
    l.red = at; at += VWAVES * MAX_ROWS * 4;
    l.misc = at; at += 64;                                                 // [0 .. 4) W_*, [4 .. 8) sixteen zero bytes (the operand of the columns without a row)
    l.total = at;
    return l;
}

#define LDSP(T, off) (reinterpret_cast<T*>(smem + (off)))
// words of a block: vector waves arrived at the barrier among themselves, at the hand-over of a phase; stop
typedef __attribute__((address_space(3))) unsigned LdsWord;             // (a generic pointer to them would be polled by flat loads, which wait for every load in flight)
__device__ __forceinline__ unsigned lds_word(int at) { return *(volatile LdsWord*)(uintptr_t)at; }
enum { W_VEC = 0, W_GO = 1, W_STOP = 3 };
__device__ __forceinline__ void arrive(int at, int lane) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane == 0) __hip_atomic_fetch_add((LdsWord*)(uintptr_t)at, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ const StepParams& args() { return step_args<StepParams>(); }

typedef float f32x2_t __attribute__((ext_vector_type(2)));

struct Ctx {
    unsigned char* smem;
    Lds l;
    int cu;
    int lane;
    unsigned tag, met;
    bool hasty;                                                             // (no time at all: the first poll in vain ends the launch)
    __device__ int first(int off) const { return (cu - off) & (CU - 1); }
    __device__ static int count(int items, int first) { return items > first ? (items - first + CU - 1) / CU : 0; }
    // a word of the block reaches `n`; false: stop
    __device__ __forceinline__ bool word(int w, unsigned n) const {
        for (;;) {
            const unsigned v = lds_word(l.misc + 4 * w), stop = lds_word(l.misc + 4 * W_STOP);
            if (__builtin_amdgcn_readfirstlane(stop)) return false;
            if (__builtin_amdgcn_readfirstlane(v) >= n) break;
            __builtin_amdgcn_s_sleep(1);
        }
        asm volatile("" ::: "memory");
        return true;
    }
    __device__ __forceinline__ void stop() const { *(volatile LdsWord*)(uintptr_t)(l.misc + 4 * W_STOP) = 1; }
    __device__ __forceinline__ bool together() {                           // the vector waves among themselves
        arrive(l.misc + 4 * W_VEC, lane);
        met += VWAVES;
        return word(W_VEC, met);
    }
    // a phase handed to the matrix waves, and its sums back.  (Barriers: matrix waves that poll a word instead take instruction fetches from the vector waves,
    // whose straight-line phases ran at 20 cycles an instruction)
    __device__ __forceinline__ void go() { arrive(l.misc + 4 * W_GO, lane); bar(); }
    __device__ __forceinline__ bool done() { bar(); return !__builtin_amdgcn_readfirstlane(lds_word(l.misc + 4 * W_STOP)); }
    // N pairs of granules (four columns each) per lane, at(i) the address of pair i, until each carries `want`; out: the four values
    template <int N, class At>
    __device__ __forceinline__ bool pairs(uint2 (&out)[N], unsigned want, At&& at) const {
        u64 t0 = 0;
        // one granule of the wave first: all of them at every poll, from every block, are as much traffic as the weights
        if (!first(reinterpret_cast<const unsigned*>(at(0)) + 1, want, t0)) return false;
        for (int n = 0;; ++n) {
            bool ok = true;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const u64* q = reinterpret_cast<const u64*>(at(i));
                const u64 lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = ok && (unsigned)(lo >> 32) == want && (unsigned)(hi >> 32) == want;
                out[i] = make_uint2((uint32_t)lo, (uint32_t)hi);
            }
            if (__all(ok)) return true;
            if (((n & 63) == 63 || hasty) && !more_time(t0)) return false;
        }
    }
    __device__ __forceinline__ bool first(const unsigned* tag_word, unsigned want, u64& t0) const {
        const unsigned long long a = (unsigned long long)tag_word;
        const unsigned* one = (const unsigned*)((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)a) | (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32)) << 32);
        for (int n = 0;; ++n) {
            unsigned v = want;
            if (lane == 0) v = __hip_atomic_load(one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_readfirstlane(v) == want) return true;
            if (((n & 63) == 63 || hasty) && !more_time(t0)) return false;
        }
    }
    __device__ __forceinline__ bool more_time(u64& t0) const { return ::more_time<StepParams>(t0, lane); }
};

// ------------------------------------------------------------------------------------------------------------------ matrix waves
template <int RING>
struct Stream {                          // this wave's weight tiles in the order it multiplies them, four to a group, through RING kilobytes of LDS
    static constexpr int GROUPS = RING / 4;
    unsigned char* smem;
    const uint2* tab;
    unsigned ring;                       // LDS bytes of slot 0
    int entries, layer, e, left, put, get, out;                            // out: groups asked for and not yet read
    int more, held;                      // held: groups in registers
    const unsigned char* at;             // per lane
    __device__ __forceinline__ void next(int lane) {
        const StepParams& p = args();
        if (e == entries) { e = 0; ++layer; }
        if (layer == p.L || entries == 0) { more = 0; left = 0; return; }
        const uint2 t = tab[e++];
        const unsigned tile = __builtin_amdgcn_readfirstlane(t.x), meta = __builtin_amdgcn_readfirstlane(t.y);
        const int role = meta & 3;
        const unsigned char* w = p.qkv.w;                                 // (values, not a reference to one of four: that would put the arguments in scratch)
        size_t step = p.qkv.layer;
        if (role == 1) { w = p.o.w; step = p.o.layer; }
        if (role == 2) { w = p.gu.w; step = p.gu.layer; }
        if (role == 3) { w = p.down.w; step = p.down.layer; }
        at = w + (size_t)layer * step + (size_t)tile * 1024 + lane * 16;
        left = meta >> 2;
    }
    // a group into the next four slots (a run is a multiple of four tiles; the offset of an LDS load moves both addresses); MOST: of this wave's loads under way, 0: any number.
    // (In assembly: the compiler would wait for every load in front of each read of LDS.  What it counts itself - the waits of its own loads - only gets stricter.)
    template <int MOST = 0>
    __device__ __forceinline__ void request(int lane) {
        if (left == 0) next(lane);
        if (!more) return;
        const unsigned to = ring + (unsigned)put * 4096u;
        if constexpr (MOST > 0)
            asm volatile("s_mov_b32 m0, %0\n\ts_waitcnt vmcnt(%2)\n\tglobal_load_lds_dwordx4 %1, off nt\n\ts_waitcnt vmcnt(%2)\n\tglobal_load_lds_dwordx4 %1, off offset:1024 nt\n\t"
                         "s_waitcnt vmcnt(%2)\n\tglobal_load_lds_dwordx4 %1, off offset:2048 nt\n\ts_waitcnt vmcnt(%2)\n\tglobal_load_lds_dwordx4 %1, off offset:3072 nt" ::"s"(to), "v"(at), "n"(MOST - 1) : "memory");
        else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\tglobal_load_lds_dwordx4 %1, off offset:1024 nt\n\t"
                     "global_load_lds_dwordx4 %1, off offset:2048 nt\n\tglobal_load_lds_dwordx4 %1, off offset:3072 nt" ::"s"(to), "v"(at) : "memory");
        at += 4096;
        left -= 4;
        ++out;
        put = put + 1 == GROUPS ? 0 : put + 1;
    }
    // the oldest group into registers
    __device__ __forceinline__ void take(bf16x8_t (&w)[4], int lane) {
        if (out == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (out == 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else if (out == 3) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
        const unsigned char* from = smem + ring + get * 4096 + lane * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const bf16x8_t*>(from + i * 1024);
        get = get + 1 == GROUPS ? 0 : get + 1;
        --out;
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
    }
    // behind a phase, until the next one is there: the ring asked for again, its oldest groups moved on into registers, their slots asked for
    __device__ __forceinline__ void fill(bf16x8_t (&pre)[AHEAD][4], int go, unsigned target, int lane) {
        for (;;) {
            if (__builtin_amdgcn_readfirstlane(lds_word(go)) >= target) break;   // the next phase is there
            if (out == GROUPS) {
                if (held == AHEAD) break;
                if (held == 0) take(pre[0], lane);
                else if (held == 1) take(pre[1], lane);
                else take(pre[AHEAD - 1], lane);
                ++held;
            }
            if (!more) break;
            request<FLIGHT>(lane);
        }
    }
};

template <int RING>
__device__ __forceinline__ void matrix_role(const Ctx& c, int wave) {
    unsigned char* smem = c.smem;
    const int R = args().rows, L = args().L;
    const StepParams& p = args();
    int lane = c.lane;
    const int off = p.qkv.items & (CU - 1);
    const int nq = Ctx::count(p.qkv.items, c.first(0)), no = Ctx::count(p.o.items, c.first(off)), ng = Ctx::count(p.gu.items, c.first(0)), nd = Ctx::count(p.down.items, c.first(off));
    const int uq = nq * p.qkv.pieces, uo = no * p.o.pieces, ug = 2 * ng * p.gu.pieces, ud = nd * p.down.pieces;
    uint2* tab = LDSP(uint2, c.l.tab) + wave * TAB;
    int n = 0;
    auto list = [&](const StepRole& r, int role, int units, int first) {
        for (int u = wave; u < units; u += MWAVES) {
            const int i = u / r.pieces, piece = u - i * r.pieces;
            const int nt = role == 2 ? 2 * (first + CU * (i >> 1)) + (i & 1) : first + CU * i;
            if (lane == 0) tab[n] = make_uint2((unsigned)(nt * r.K_tiles + piece * r.len), (unsigned)(role | r.len << 2));
            ++n;
        }
    };
    list(p.qkv, 0, uq, c.first(0));
    list(p.o, 1, uo, c.first(off));
    list(p.gu, 2, ug, c.first(0));
    list(p.down, 3, ud, c.first(off));
    wave_lds_fence();
    Stream<RING> st{smem, tab, (unsigned)__builtin_amdgcn_readfirstlane(c.l.ring + wave * RING * 1024), n, 0, 0, 0, 0, 0, 0, 1, 0, nullptr};

    bf16x8_t pre[AHEAD][4];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) pre[i][j] = (bf16x8_t){0, 0, 0, 0, 0, 0, 0, 0};
    const int col = lane & 15, g4 = lane >> 4;
    const bool on = col < R;
    unsigned target = 0;
    for (int li = 0; li < L; ++li) {
        for (int ph = 0; ph < 4; ++ph) {
            if (li + ph) bar();                                            // (behind the values of the phase before, whose stores would stand in line after the requests)
            target += VWAVES;
            st.fill(pre, c.l.misc + 4 * W_GO, target, lane);
            bar();
            if (__builtin_amdgcn_readfirstlane(lds_word(c.l.misc + 4 * W_STOP))) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); return; }
            const StepParams& p = args();
            const int units = ph == 0 ? uq : ph == 1 ? uo : ph == 2 ? ug : ud;
            const int pieces = ph == 0 ? p.qkv.pieces : ph == 1 ? p.o.pieces : ph == 2 ? p.gu.pieces : p.down.pieces;
            const int per = (ph == 0 ? p.qkv.len : ph == 1 ? p.o.len : ph == 2 ? p.gu.len : p.down.len) >> 2;      // groups a unit
            int rest = units > wave ? (units - wave + MWAVES - 1) / MWAVES * per : 0, u = wave, left = 0;
            // x from LDS: [k-tile][quarter][row][8]
            unsigned xa = 0;
            const unsigned step = on ? 64 * R : 0;
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
            auto group = [&](const bf16x8_t (&w)[4], const bf16x8_t (&x)[4]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[i], acc, 0, 0, 0);
                --rest;
                if (--left == 0) {
                    if (on) *reinterpret_cast<f32x4_t*>(smem + c.l.part + ((size_t)u * R + col) * 64 + g4 * 16) = acc;
                    u += MWAVES;
                }
            };
            auto operand = [&](bf16x8_t (&x)[4]) {
                if (left == 0) {
                    left = per;
                    acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                    xa = on ? c.l.xs + u % pieces * per * 256 * R + (g4 * R + col) * 16 : c.l.misc + 16;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) { x[i] = *reinterpret_cast<const bf16x8_t*>(smem + xa); xa += step; }
            };
            int used = 0;
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                if (i < st.held && rest > 0) {
                    bf16x8_t x[4];
                    operand(x);
                    group(pre[i], x);
                    used = i + 1;
                }
            }
            // (what is left of the held groups belongs to the next phase)
            if (used) {
#pragma unroll
                for (int s = 1; s < AHEAD; ++s) {
                    if (used == s) {
#pragma unroll
                        for (int i = 0; i + s < AHEAD; ++i)
#pragma unroll
                            for (int j = 0; j < 4; ++j) pre[i][j] = pre[i + s][j];
                    }
                }
                st.held -= used;
            }
            while (rest > 0) {
                bf16x8_t x[4], w[4];
                if (rest > st.out && st.out < Stream<RING>::GROUPS) st.request(lane);   // (the slots of the group before are free; nothing asked for: at least this one)
                operand(x);
                st.take(w, lane);
                group(w, x);
            }
            bar();
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ------------------------------------------------------------------------------------------------------------------ vector waves
__device__ __forceinline__ uint32_t bf_pack(float a, float b) { return (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16); }

// residual stream of one edge -> RMSNorm (k_glue_cpt's columns, sums and rounding) -> sink(row, first of four columns, values)
template <class Sink>
__device__ __forceinline__ bool norm_rows(Ctx& c, const unsigned char* hx, const bf16_t* wn, unsigned want, int vt, int vw, Sink&& sink) {
    const StepParams& p = args();
    unsigned char* smem = c.smem;
    float* red = LDSP(float, c.l.red);
    const int R = p.rows, lane = c.lane;
    uint2 wq[CPT];
#pragma unroll
    for (int g = 0; g < CPT; ++g) wq[g] = *reinterpret_cast<const uint2*>(wn + 4 * (vt + g * VT));
    uint2 hq[MAX_ROWS][CPT];
    bool ok = true;
#pragma unroll
    for (int r = 0; r < MAX_ROWS; ++r) {
#pragma unroll
        for (int g = 0; g < CPT; ++g) hq[r][g] = make_uint2(0, 0);
        if (r < R) ok = ok && c.pairs(hq[r], want, [&](int g) { return hx + ((size_t)r * (p.d >> 2) + vt + g * VT) * 16; });
    }
#pragma unroll
    for (int r = 0; r < MAX_ROWS; ++r) {
        if (r >= R) break;
        float ss = 0.0f;
#pragma unroll
        for (int g = 0; g < CPT; ++g) {
            const float hn[4] = {bf_lo(hq[r][g].x), bf_hi(hq[r][g].x), bf_lo(hq[r][g].y), bf_hi(hq[r][g].y)};
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += hn[e] * hn[e];
        }
        ss = wave_sum_dpp(ss);
        if (lane == 0) red[r * VWAVES + vw] = ss;
    }
    if (!ok) c.stop();
    if (!c.together()) return false;
#pragma unroll
    for (int r = 0; r < MAX_ROWS; ++r) {
        if (r >= R) break;
        float tot = 0.0f;
#pragma unroll
        for (int i = 0; i < VWAVES; ++i) tot += red[r * VWAVES + i];
        const float inv = 1.0f / sqrtf(tot / (float)p.d + p.eps);
#pragma unroll
        for (int g = 0; g < CPT; ++g) {
            const float hn[4] = {bf_lo(hq[r][g].x), bf_hi(hq[r][g].x), bf_lo(hq[r][g].y), bf_hi(hq[r][g].y)};
            const float wv[4] = {bf_lo(wq[g].x), bf_hi(wq[g].x), bf_lo(wq[g].y), bf_hi(wq[g].y)};
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = wv[e] * bf16_round_f32(hn[e] * inv);
            sink(r, 4 * (vt + g * VT), make_uint2(bf_pack(x[0], x[1]), bf_pack(x[2], x[3])), hq[r][g]);
        }
    }
    return true;
}

// decode attention of one (row, kv head): k_attn_decode2's arithmetic, its eight waves' tiles and partial sums kept apart on four waves
__device__ __forceinline__ bool attention(Ctx& c, const unsigned char* xq, unsigned char* xa, int li, unsigned want, int vt, int vw) {
    constexpr int D = 128;
    const StepParams& p = args();
    unsigned char* smem = c.smem;
    const int lane = c.lane, b = c.cu / p.Hkv, kvh = c.cu - b * p.Hkv, G = p.H / p.Hkv, h = lane & 15, g4 = lane >> 4;
    float* strip = LDSP(float, c.l.strip) + (size_t)vw * (G + 3) * D;
    float *sO = LDSP(float, c.l.so), *sm = LDSP(float, c.l.sm), *sl = sm + VIRT * 16;
    const int pos = p.pos[b];
    const bool live = p.active[b] != 0;
    const int kv_len = pos + 1, n_tiles = (kv_len + 31) >> 5, new_tile = pos >> 5;
    bf16_t* kc = p.kcache + p.kv_layer * li + ((size_t)(b * p.Hkv + kvh) * p.Smax) * D;
    bf16_t* vt_ = p.vcache + p.kv_layer * li + ((size_t)(b * p.Hkv + kvh) * D) * p.Smax;
    f32x4_t rc[2][2], rs[2][2];
    {
        const float* ct = p.rope_cos + (size_t)pos * (D / 2) + g4 * 8;
        const float* st = p.rope_sin + (size_t)pos * (D / 2) + g4 * 8;
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int j = 0; j < 2; ++j) { rc[k][j] = *reinterpret_cast<const f32x4_t*>(ct + k * 32 + j * 4); rs[k][j] = *reinterpret_cast<const f32x4_t*>(st + k * 32 + j * 4); }
    }
    bf16x8_t ka[2][4], vb[8];
    auto load_k = [&](int tile) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ka[i >> 2][i & 3] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(kc + (size_t)tile * 32 * D) + i * 64 + lane);
    };
    auto load_v = [&](int tile) {
#pragma unroll
        for (int i = 0; i < 8; ++i) vb[i] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(vt_ + (size_t)tile * 32 * D) + i * 64 + lane);
    };
    // tiles of this wave: vw, vw + 8, .. (virtual wave vw), then vw + 4, vw + 12, .. (virtual wave vw + 4)
    const int t_first = vw < n_tiles ? vw : 0;
    load_k(t_first);
    uint2 qkv[3];
    const bool ok = c.pairs(qkv, want, [&](int i) {
        int u = lane + 64 * i;
        u = u < (G + 2) * D / 4 ? u : 0;
        const int e0 = u * 4, hh = e0 / D, dd = e0 - hh * D, n = (hh < G ? kvh * G + hh : hh == G ? p.H + kvh : p.H + p.Hkv + kvh) * D + dd;
        return xq + ((size_t)b * (p.H + 2 * p.Hkv) * D + n) * 4;
    });
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int u = lane + 64 * i;
        if (u < (G + 2) * D / 4) *reinterpret_cast<f32x4_t*>(strip + 4 * u) = (f32x4_t){bf_lo(qkv[i].x), bf_hi(qkv[i].x), bf_lo(qkv[i].y), bf_hi(qkv[i].y)};
    }
    wave_lds_fence();
    bf16_t* kro = reinterpret_cast<bf16_t*>(strip + (G + 2) * D);
    auto rope_row = [&](int row, bf16x8_t (&out)[4]) {
        f32x4_t x[4][2];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k][0] = *reinterpret_cast<const f32x4_t*>(strip + row * D + k * 32 + g4 * 8);
            x[k][1] = *reinterpret_cast<const f32x4_t*>(strip + row * D + k * 32 + g4 * 8 + 4);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x1 = x[k][e >> 2][e & 3], x2 = x[k + 2][e >> 2][e & 3];
                const float cs = rc[k][e >> 2][e & 3], sn = rs[k][e >> 2][e & 3];
                out[k][e] = (short)f32_to_bf16(fmaf(x1, cs, -(x2 * sn)));
                const float a = p.schedule2 ? x2 * cs : x1 * sn;                              // the product that k_attn_decode2, or k_attn_decode, rounds
                out[k + 2][e] = (short)f32_to_bf16(fmaf(p.schedule2 ? x1 : x2, p.schedule2 ? sn : cs, a));
            }
    };
    bf16x8_t qf[4];
    rope_row(h < G ? h : G - 1, qf);
    if (h >= G) {
#pragma unroll
        for (int k = 0; k < 4; ++k) qf[k] = (bf16x8_t){0, 0, 0, 0, 0, 0, 0, 0};
    }
    {
        bf16x8_t kn[4];
        rope_row(G, kn);
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<bf16x8_t*>(kro + k * 32 + g4 * 8) = kn[k];
    }
    wave_lds_fence();
    load_v(t_first);
    const int pr = pos & 31, prow = ((pr >> 3) << 2) | (pr & 3), phalf = (pr >> 2) & 1;
    f32x4_t O[D / 16];
    float m_run, l_run;
    if (live) {
        for (int half = 0; half < 2; ++half) {
            const int vwave = vw + 4 * half;
            if (vwave >= n_tiles) break;                                    // (the chain's waves without a tile add nothing)
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) O[dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            m_run = -INFINITY; l_run = 0.0f;
            for (int tile = vwave; tile < n_tiles; tile += VIRT) {
                const int nxt = tile + VIRT < n_tiles ? tile + VIRT : half == 0 && vw + 4 < n_tiles ? vw + 4 : -1;
                if (tile == new_tile) {                                    // the new key and value join, and go to the caches
                    if ((lane & 15) == prow) {
                        bf16x8_t* dst = reinterpret_cast<bf16x8_t*>(kc) + ((size_t)new_tile * 2 + phalf) * (D / 32) * 64 + lane;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const bf16x8_t kn = *reinterpret_cast<const bf16x8_t*>(kro + k * 32 + g4 * 8);
                            if (phalf) ka[1][k] = kn; else ka[0][k] = kn;
                            dst[k * 64] = kn;
                        }
                    }
                    if ((lane >> 4) == (pr >> 3)) {
#pragma unroll
                        for (int dt = 0; dt < 8; ++dt) {
                            const bf16_t vn = f32_to_bf16(strip[(G + 1) * D + dt * 16 + (lane & 15)]);
#pragma unroll
                            for (int e = 0; e < 8; ++e)
                                if (e == (pr & 7)) vb[dt][e] = (short)vn;
                            vt_[(((size_t)new_tile * (D / 16) + dt) * 64 + lane) * 8 + (pr & 7)] = vn;
                        }
                    }
                }
                const int base = tile * 32;
                f32x4_t S0 = (f32x4_t){0.f, 0.f, 0.f, 0.f}, S1 = S0;
#pragma unroll
                for (int k = 0; k < D / 32; ++k) {
                    S0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[0][k], qf[k], S0, 0, 0, 0);
                    S1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[1][k], qf[k], S1, 0, 0, 0);
                }
                if (nxt >= 0) load_k(nxt);
                float sc[8];
                float mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float v = (e < 4 ? S0[e] : S1[e - 4]) * p.scale;
                    v = (base + g4 * 8 + e < kv_len) ? v : -INFINITY;
                    sc[e] = v;
                    mx = fmaxf(mx, v);
                }
                mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                float m_new = fmaxf(m_run, mx);
                float alpha = __expf(m_run - m_new);
                float psum = 0.0f;
                bf16x8_t ph, pl;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float pe = __expf(sc[e] - m_new);
                    psum += pe;
                    bf16_t hi = f32_to_bf16(pe);
                    bf16_t lo = f32_to_bf16(pe - bf16_to_f32(hi));
                    ph[e] = (short)hi;
                    pl[e] = (short)lo;
                }
                l_run = l_run * alpha + psum;
                m_run = m_new;
                float ar[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, g4 * 4 + r, 64);
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt) {
                    f32x4_t o = O[dt];
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] *= ar[r];
                    o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vb[dt], o, 0, 0, 0);
                    o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vb[dt], o, 0, 0, 0);
                    O[dt] = o;
                }
                if (nxt >= 0) load_v(nxt);
            }
            l_run += __shfl_xor(l_run, 16, 64);
            l_run += __shfl_xor(l_run, 32, 64);
            if (g4 == 0) { sm[vwave * 16 + h] = m_run; sl[vwave * 16 + h] = l_run; }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int head = g4 * 4 + r;
                if (head < G) {
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) sO[((size_t)vwave * G + head) * D + dt * 16 + h] = O[dt][r];
                }
            }
        }
    }
    if (!ok) c.stop();
    if (!c.together()) return false;
    if (live) {
        for (int i = vt; i < G * D / 2; i += VT) {
            const int head = 2 * i / D, d0 = 2 * i - head * D;
            float M = -INFINITY;
#pragma unroll
            for (int w = 0; w < VIRT; ++w) M = w < n_tiles ? fmaxf(M, sm[w * 16 + head]) : M;
            float num[2] = {0.0f, 0.0f}, den = 0.0f;
#pragma unroll
            for (int w = 0; w < VIRT; ++w) {
                if (w >= n_tiles) break;
                const float f = __expf(sm[w * 16 + head] - M);
                num[0] += f * sO[((size_t)w * G + head) * D + d0];
                num[1] += f * sO[((size_t)w * G + head) * D + d0 + 1];
                den += f * sl[w * 16 + head];
            }
            granule(xa + ((size_t)b * p.H * D + (kvh * G + head) * D + d0) * 4, bf_pack(num[0] / den, num[1] / den), want);
        }
    } else {                                                               // (a row that has ended: zeros, so that nobody waits for it)
        for (int i = vt; i < G * D / 2; i += VT) granule(xa + ((size_t)b * p.H * D + kvh * G * D + 2 * i) * 4, 0, want);
    }
    return c.together();                                                   // (nobody may write the operand over the partial sums before all have read them)
}

// Sum of a column tile's pieces, two columns of a row, in the chain's order: the waves of a slab, then the slabs.  (One copy: the instruction cache holds the
// whole layer or every phase begins with a miss per line.)
__device__ __attribute__((noinline)) float2 pieces_total(int at, int step, int pieces, int ksb) {
    typedef __attribute__((address_space(3))) const f32x2_t Lds2;
    f32x2_t v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = *(Lds2*)(uintptr_t)(at + min(i, pieces - 1) * step);
    float2 s = make_float2(0.0f, 0.0f), t = s;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i < pieces) {
            const bool head = (i & (ksb - 1)) == 0, tail = ((i + 1) & (ksb - 1)) == 0;
            t.x = head ? v[i][0] : t.x + v[i][0];
            t.y = head ? v[i][1] : t.y + v[i][1];
            s.x = tail ? s.x + t.x : s.x;
            s.y = tail ? s.y + t.y : s.y;
        }
    }
    return s;
}

__device__ __forceinline__ void vector_role(Ctx c, const int vw) {
    const StepParams& p0 = args();
    const int L = p0.L, d = p0.d, R = p0.rows;
    unsigned char* smem = c.smem;
    int lane, vt, r, cp;                                                    // r, cp: row and pair of columns when pieces are combined
    bool on;
    // addresses are made anew in each phase: kept over the layer they are more than there are registers
    auto fresh = [&]() {
        asm volatile("" : "+v"(c.lane));
        lane = c.lane; vt = vw * 64 + lane; r = lane >> 3; cp = lane & 7; on = r < R;
    };
    fresh();
    const int off = p0.qkv.items & (CU - 1), fq = c.first(0), fo = c.first(off);
    const int nq = Ctx::count(p0.qkv.items, fq), no = Ctx::count(p0.o.items, fo), ng = Ctx::count(p0.gu.items, fq), nd = Ctx::count(p0.down.items, fo);
    const bool attn = c.cu < R * p0.Hkv;
    const Layout ex = exch_layout(d, 32 * p0.down.K_tiles, p0.H, p0.Hkv, 128, R);
    auto to_lds = [&](int row, int k, uint2 x) { *reinterpret_cast<uint2*>(smem + c.l.xs + (k >> 5) * 64 * R + (((k & 31) >> 3) * R + row) * 16 + ((k & 7) >> 2) * 8) = x; };
    auto total = [&](int u0, const StepRole& ro) { return pieces_total(c.l.part + (u0 * R + r) * 64 + cp * 8, 64 * R, ro.pieces, ro.ksb); };
    // half layers: the attention's, the MLP's, and behind the last one the final norm
    for (int hf = 0; hf <= 2 * L; ++hf) {
        const int li = hf >> 1, half = hf & 1;
        if (hf == 2 * L && c.cu) return;
        const unsigned want = c.tag + li + 1;
        unsigned char* xl = args().exch + (size_t)ex.layer * li;
        const unsigned char* hin = half ? xl + ex.h1 : xl - ex.layer + ex.h2;
        fresh();
        if (hf == 0) {
            const StepParams& p = args();
            const int MT = p.Mpad >> 4;
            for (int i = vt; i < R * (d >> 2); i += VT) {
                const int row = i / (d >> 2), k = 4 * (i - row * (d >> 2));
                to_lds(row, k, *reinterpret_cast<const uint2*>(p.x0 + xpk_index(row, k, MT)));
            }
        } else {
            const bool last = hf == 2 * L;
            auto sink = [&](int row, int k, uint2 x, uint2 hv) {
                if (!last) { to_lds(row, k, x); return; }
                const StepParams& p = args();
                *reinterpret_cast<uint2*>(p.x_out + xpk_index(row, k, p.Mpad >> 4)) = x;
                *reinterpret_cast<uint2*>(p.h_out + (size_t)row * d + k) = hv;
            };
            if (!norm_rows(c, hin, args().norms + (size_t)hf * d, want - 1 + half, vt, vw, sink)) return;
            if (last) {                                                    // every block has passed its last edge but one: the tag base may move
                if (vt == 0) args().sync[SYNC_TAG] = c.tag + L + 1;
                return;
            }
        }
        c.go();
        if (!c.done()) return;
        fresh();
        const int n = half ? nd : no;
        uint32_t old = 0;
        if (!half) {
            for (int i = vw; i < nq; i += VWAVES) {
                const StepParams& p = args();
                const int nt = fq + CU * i;
                if (on) {
                    const float2 s = total(i * p.qkv.pieces, p.qkv);
                    granule(xl + ex.q + ((size_t)r * p.qkv.items * 8 + nt * 8 + cp) * 8, bf_pack(s.x, s.y), want);
                }
            }
            if (!attn) bar();
            fresh();
            if (attn) { if (!attention(c, xl + ex.q, xl + ex.a, li, want, vt, vw)) return; }
            if (attn) bar();                                                // (their requests would be in front of the attention's)
            fresh();
            bool ok = true;
            for (int row = 0; row < R; ++row) {
                uint2 v[CPT];
                ok = ok && c.pairs(v, want, [&](int g) { return xl + ex.a + ((size_t)row * (d >> 2) + vt + g * VT) * 16; });
#pragma unroll
                for (int g = 0; g < CPT; ++g) to_lds(row, 4 * (vt + g * VT), v[g]);
            }
            if (!ok) { c.stop(); return; }
        } else {
            for (int i = vw; i < ng; i += VWAVES) {
                const StepParams& p = args();
                const int pr = fq + CU * i;
                if (on) {
                    const float2 g = total(2 * i * p.gu.pieces, p.gu), u = total((2 * i + 1) * p.gu.pieces, p.gu);
                    const float gg[2] = {bf16_round_f32(g.x), bf16_round_f32(g.y)}, uu[2] = {bf16_round_f32(u.x), bf16_round_f32(u.y)};
                    float a[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float sg = bf16_round_f32(1.0f / (1.0f + __expf(-gg[e])));
                        a[e] = bf16_round_f32(gg[e] * sg) * uu[e];
                    }
                    granule(xl + ex.act + ((size_t)r * p.gu.items * 8 + pr * 8 + cp) * 8, bf_pack(a[0], a[1]), want);
                }
            }
            bar();
            fresh();
            const int quads = 4 * args().gu.items;                          // four columns each
            if (nd) {
                bool ok = true;
                for (int row = 0; row < R; ++row)
                    for (int i0 = 0; i0 < quads; i0 += 4 * VT) {
                        uint2 v[4];
                        ok = ok && c.pairs(v, want, [&](int g) { return xl + ex.act + ((size_t)row * quads + min(i0 + vt + g * VT, quads - 1)) * 16; });
#pragma unroll
                        for (int g = 0; g < 4; ++g) to_lds(row, 4 * min(i0 + vt + g * VT, quads - 1), v[g]);
                    }
                if (!ok) { c.stop(); return; }
            }
        }
        // this lane's pair of columns of the residual stream as the block has seen it arrive
        if (on && vw < n) {
            const int nt = fo + CU * vw;
            old = hf == 0 ? *reinterpret_cast<const uint32_t*>(args().h0 + (size_t)r * d + nt * 16 + cp * 2)
                          : (uint32_t)__hip_atomic_load(reinterpret_cast<const u64*>(hin + ((size_t)r * (d >> 1) + nt * 8 + cp) * 8), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        c.go();
        if (!c.done()) return;
        fresh();
        if (on && vw < n) {
            const StepParams& p = args();
            const int nt = fo + CU * vw;
            const float2 s = half ? total(vw * p.down.pieces, p.down) : total(vw * p.o.pieces, p.o);
            granule(xl + (half ? ex.h2 : ex.h1) + ((size_t)r * (d >> 1) + nt * 8 + cp) * 8, bf_pack(bf_lo(old) + bf16_round_f32(s.x), bf_hi(old) + bf16_round_f32(s.y)), want);
        }
        if (hf + 1 < 2 * L) bar();
    }
}

// One block a compute unit (its LDS sees to that); all of them have to be resident: nobody leaves before every block's values have come.
template <int RING>
__global__ void __launch_bounds__(THREADS, 1) k_step_layers(StepParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int cu = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = p.H / p.Hkv, R = p.rows;
    const int uq = (p.qkv.items + CU - 1) / CU * p.qkv.pieces, ug = 2 * ((p.gu.items + CU - 1) / CU) * p.gu.pieces, ud = p.down.pieces, uo = p.o.pieces;
    const int mu = max(max(uq, ug), max(ud, uo));
    Ctx c{smem, lds_layout(RING, 32 * max(p.qkv.K_tiles, max(p.o.K_tiles, p.down.K_tiles)), R, G, mu), cu, lane, p.sync[SYNC_TAG], 0, p.limit == 0};
    if (threadIdx.x < 16) LDSP(int, c.l.misc)[threadIdx.x] = threadIdx.x == W_STOP && __hip_atomic_load(p.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ? 1 : 0;
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(lds_word(c.l.misc + 4 * W_STOP))) {
        if (wave < MWAVES) matrix_role<RING>(c, wave);
        else vector_role(c, wave - MWAVES);
    }
}
int max_units(const StepParams& p) {
    const int uq = (p.qkv.items + CU - 1) / CU * p.qkv.pieces, ug = 2 * ((p.gu.items + CU - 1) / CU) * p.gu.pieces;
    return std::max(std::max(uq, ug), std::max(p.o.pieces, p.down.pieces));
}
int k_max(const StepParams& p) { return 32 * std::max(p.qkv.K_tiles, std::max(p.o.K_tiles, p.down.K_tiles)); }

constexpr int LDS_MAX = 160 * 1024;
int lds_bytes(const StepParams& p, int ring) { return lds_layout(ring, k_max(p), p.rows, p.H / p.Hkv, max_units(p)).total; }
// kilobytes of ring a matrix wave: what fits (one row 16; two rows' operand of the down projection leaves 12)
int ring_of(const StepParams& p) { return lds_bytes(p, 16) <= LDS_MAX ? 16 : lds_bytes(p, 12) <= LDS_MAX ? 12 : 0; }
}

size_t step_exch_bytes(const StepShape& s) { return (size_t)exch_layout(s.d, s.ff, s.H, s.Hkv, s.D, s.rows).layer * s.L; }

bool step_ok(const StepShape& s, const StepParams& p, int device) {
    // widths: RMSNorm's columns are dealt as k_glue_cpt deals them; attention's heads as k_attn_decode2 takes them
    if (s.rows < 1 || s.rows > MAX_ROWS || s.D != 128 || s.H % s.Hkv || s.H / s.Hkv > 4 || s.d != 4 * CPT * VT || s.H * s.D != s.d || s.rows * s.Hkv > CU || s.ff % 16) return false;
    const StepRole* roles[4] = {&p.qkv, &p.o, &p.gu, &p.down};
    int entries = 0;
    for (int i = 0; i < 4; ++i) {
        const StepRole& r = *roles[i];
        if (r.pieces < 1 || r.pieces > 16 || r.ksb < 1 || (r.ksb & (r.ksb - 1)) || r.pieces % r.ksb || r.len % 4 || r.pieces * r.len != r.K_tiles) return false;
        entries += ((r.items + CU - 1) / CU * (i == 2 ? 2 : 1) * r.pieces + MWAVES - 1) / MWAVES;
    }
    if (p.o.items != p.down.items || p.o.items > CU || entries > TAB || !ring_of(p)) return false;             // one tile of the residual stream a block
    int cus = 0, lds = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device) != hipSuccess) return false;
    if (cus < CU || lds < LDS_MAX) return false;
    for (auto f : {reinterpret_cast<const void*>(&k_step_layers<16>), reinterpret_cast<const void*>(&k_step_layers<12>)})
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX) != hipSuccess) { (void)hipGetLastError(); return false; }
    return true;
}

void launch_step(const StepParams& p, hipStream_t s) {
    const int ring = ring_of(p), lds = lds_bytes(p, ring);
    if (ring == 16) hipLaunchKernelGGL((k_step_layers<16>), dim3(CU), dim3(THREADS), lds, s, p);
    else hipLaunchKernelGGL((k_step_layers<12>), dim3(CU), dim3(THREADS), lds, s, p);
}

bool step_was_late(const unsigned* sync, StepPause& pause, const char* what) {
    unsigned late = 0;
    HIP_CHECK(copy_now(&late, sync + SYNC_LATE, sizeof(late), hipMemcpyDeviceToHost));
    if (!late) return false;
    pause.late();
    fprintf(stderr, "mi_speech: a %s step waited in vain for compute units (held from outside this library); its request runs again on the launch chain, and so do the handle's next %d\n", what,
            pause.skip);
    return true;
}
