// codec_f32.hip - the exact-f32 dense contractions of the codecs: Y[b][m][n] = epilogue(sum_k A[m][k] act(X[b][row(k)][n + shift(k)])) on f32 MFMA.
//
// 1x1 convolutions (plain, GELU, residual with optional Snake in front, NoiseBlock) and dense k-tap convolutions without an activation (the encoders'
// strided convolutions over a phase-split tensor).  The k order is: 16 input channels, within them the taps, within a tap the channels.
// v_mfma_f32 adds its products one after the other in k order (32x32x2, 16x16x4 and a chain of fmaf give the same bits: measured over random
// operands), so EVERY tile shape below returns the same bits and the launcher is free to pick one by the number of blocks it gives.  Convolutions of K >= 1024 add four
// partial sums, in every form that they may take:
//
//   wide   128 x 64 (M <= 64: 64 x 128), 4 waves of 64 x 32 on 32x32x2, 16 k per staged chunk, three blocks per compute unit: a block's loads and its
//          epilogue hide behind the others' products.  Bound: 2.4 GB for 256 x 24576 outputs over K = 256 with residual, 32 rows: 1.18 ms of 1.34 ms
//          before (64 x 128 tiles, two barriers per chunk, residual rows one by one); 128 x 128 tiles at two blocks per unit: 1.36 ms.
//   small  32 x 32, 4 waves of one 16x16x4 tile, four chunks of 64 k in flight at once (a short K is ONE memory round trip).  Bound: latency.
//          512 x 384 outputs over K = 512 with residual: 45 -> 7.5 us.
//   split  32 x 16, the four waves a quarter of a long K each (k_codec_gemm_split).
//
// One barrier per chunk (two LDS buffers): chunk c + 1 goes from registers to LDS and chunk c + 1 + PF is requested before chunk c is multiplied.
// Blocks are dealt to the XCDs by id mod 8: an XCD takes a CONTIGUOUS range of column tiles, all row tiles of a column tile in a row.  Its L2 holds the
// X tile for the row tiles, and its 16 channels (256 bytes apart) are all in use - with every eighth 512-byte tile on one XCD two of them serve it.
#include "common.h"
#include "codec_kernels.h"

#include <algorithm>
#include <type_traits>


struct F32Tiles { int nt, mt, npx, taps; };      // column tiles, row tiles, column tiles per XCD
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));       // four columns of a row at any column: global loads need 4-byte alignment only

// One tile.  WM x WN waves; a wave holds TM x TN MFMA tiles of MS x MS (MS = 32 or 16); BK k per chunk; PF chunks requested ahead.
// IN: the tile lies inside the output, its columns at every tap inside the input, M is a multiple of 4, the channels of 16 and the k units of the chunk -
// nothing to clamp or mask.  Otherwise every element is clamped when it is loaded and masked when it is put into LDS.
// OFF: the type of an offset inside the tile's rows (see launch_f32).  QUARTERS: four partial sums (codec_quarters), the accumulators added to the total between them.
template <int MODE, bool SNAKE, int MS, int WM, int WN, int TM, int TN, int BK, int PF, bool IN, typename OFF, bool QUARTERS>
__device__ __forceinline__ void codec_gemm_tile(const GemmParams& p, int T, int n0, int m0, int b, float* As, float* Xs, const float* __restrict__ pX, const float* __restrict__ pR,
                                                float* __restrict__ pY, const float* __restrict__ pbias, const float* __restrict__ pscale, const float* __restrict__ pAT) {
    constexpr int BM = WM * TM * MS, BN = WN * TN * MS, KS = MS == 32 ? 2 : 4;
    constexpr int LA = MS == 32 ? BM : BM + 16, LX = MS == 32 ? BN : BN + 16;      // (16x16x4 reads four k rows at once: 16 banks apart)
    constexpr int NA = BK * BM / 4 / 256, NX = BK * BN / 4 / 256;                  // float4 of A and of X per thread
    static_assert(NA * 256 * 4 == BK * BM && NX * 256 * 4 == BK * BN && BK % 16 == 0, "whole pieces");
    typedef typename std::conditional<MS == 32, f32x16_t, f32x4_t>::type acc_t;
    constexpr int NR = MS == 32 ? 16 : 4;
    constexpr bool PRE = MS == 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    constexpr bool taps = MODE == GEMM_TAPS;
    const int Cin = taps ? p.Cin : p.K;
    const int units = (Cin + 15) / 16 * T, nchunks = (units + BK / 16 - 1) / (BK / 16);
    const float* Xb = pX + (size_t)b * Cin * p.ldx;
    // piece i of a thread (PW pieces per k row) of chunk c: its unit of 16 k, channel block and tap are scalar (a wave's 64 pieces lie inside one unit)
    auto unit = [&](int c, int i, auto pw, int& c16, int& tap) {
        constexpr int PW = decltype(pw)::value;
        static_assert(64 / PW <= 16, "a wave's pieces inside one unit");
        const int u = c * (BK / 16) + (((wave * 64 + i * 256) / PW) >> 4);
        const int uc = min(u, units - 1), cc = taps ? uc / T : uc;
        tap = taps ? uc - cc * T : 0;
        c16 = cc * 16;
        return u < units;
    };
    const std::integral_constant<int, BM / 4> pwa{};
    const std::integral_constant<int, BN / 4> pwx{};
    // Addresses are a scalar base plus an offset (32 bits unless rows are very long); loads are unconditional (a guarded load becomes a branch whose join waits for everything in flight)
    auto at = [](const float* base, OFF off) { return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off); };
    float4 ra[PF][NA], rx[PF][NX];
    auto load = [&](int c, int slot) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int m = m0 + ((tid + i * 256) & (BM / 4 - 1)) * 4, r = ((tid + i * 256) / (BM / 4)) & 15;
            int c16, tap;
            unit(c, i, pwa, c16, tap);
            const float* base = pAT + (size_t)(tap * Cin + c16) * p.M;
            if constexpr (IN) ra[slot][i] = *reinterpret_cast<const float4*>(at(base, 4u * (uint32_t)(r * p.M + m)));
            else {
                const uint32_t row = (uint32_t)(min(r, Cin - 1 - c16) * p.M);
                ra[slot][i] = make_float4(base[row + min(m, p.M - 1)], base[row + min(m + 1, p.M - 1)], base[row + min(m + 2, p.M - 1)], base[row + min(m + 3, p.M - 1)]);
            }
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int nl = ((tid + i * 256) & (BN / 4 - 1)) * 4, r = ((tid + i * 256) / (BN / 4)) & 15;
            int c16, tap;
            unit(c, i, pwx, c16, tap);
            const int sh = taps ? tap * p.dil - p.pad : 0;
            if constexpr (IN) {
                const f32x4u_t v = *reinterpret_cast<const f32x4u_t*>(at(Xb + (int64_t)c16 * p.ldx + n0 + sh, 4 * ((OFF)r * p.ldx + nl)));
                rx[slot][i] = make_float4(v[0], v[1], v[2], v[3]);
            } else {
                const float* row = Xb + (int64_t)(c16 + min(r, Cin - 1 - c16)) * p.ldx;
                const int n = n0 + nl + sh;
                auto in = [&](int e) { return row[min(max(n + e, p.x_lo), p.Tin - 1)]; };
                rx[slot][i] = make_float4(in(0), in(1), in(2), in(3));
            }
        }
    };
    auto put = [&](int c, int slot, int buf) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int idx = tid + i * 256, rr = idx / (BM / 4), ml = (idx & (BM / 4 - 1)) * 4, m = m0 + ml;
            float4 v = ra[slot][i];
            if constexpr (!IN) {
                int c16, tap;
                const bool ok = unit(c, i, pwa, c16, tap) && c16 + (rr & 15) < Cin;
                v = make_float4(ok && m < p.M ? v.x : 0.f, ok && m + 1 < p.M ? v.y : 0.f, ok && m + 2 < p.M ? v.z : 0.f, ok && m + 3 < p.M ? v.w : 0.f);
            }
            *reinterpret_cast<float4*>(As + buf * (BK * LA) + rr * LA + ml) = v;
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int idx = tid + i * 256, rr = idx / (BN / 4), nl = (idx & (BN / 4 - 1)) * 4;
            int c16, tap;
            const bool in = unit(c, i, pwx, c16, tap);
            float4 v = rx[slot][i];
            if constexpr (!IN) {
                const bool ok = in && c16 + (rr & 15) < Cin;
                const int n = n0 + nl + (taps ? tap * p.dil - p.pad : 0);
                auto keep = [&](float x, int e) { return ok && n + e >= p.x_lo && n + e < p.Tin ? x : 0.0f; };
                v = make_float4(keep(v.x, 0), keep(v.y, 1), keep(v.z, 2), keep(v.w, 3));
            }
            if constexpr (SNAKE) {
                const int ch = min(c16 + (rr & 15), Cin - 1);
                const float a = p.alpha[ch], al = p.ralpha[ch];
                v = make_float4(mis_snake(v.x, a, al), mis_snake(v.y, a, al), mis_snake(v.z, a, al), mis_snake(v.w, a, al));      // snake(0) = 0 keeps the zero pad
            }
            *reinterpret_cast<float4*>(Xs + buf * (BK * LX) + rr * LX + nl) = v;
        }
    };
    acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[i][j][r] = 0.0f;
    auto math = [&](int buf) {
        const float* a0 = As + buf * (BK * LA) + (MS == 32 ? lane >> 5 : lane >> 4) * LA + wm * TM * MS + (lane & (MS - 1));
        const float* x0 = Xs + buf * (BK * LX) + (MS == 32 ? lane >> 5 : lane >> 4) * LX + wn * TN * MS + (lane & (MS - 1));
        constexpr int FD = MS == 32 ? 2 : 4;             // fragments are read FD - 1 steps ahead (an LDS read is 3 to 4 of the small tile's steps)
        float av[FD][TM], xv[FD][TN];
        auto frag = [&](int kk, int h) {
#pragma unroll
            for (int i = 0; i < TM; ++i) av[h][i] = a0[kk * LA + i * MS];
#pragma unroll
            for (int j = 0; j < TN; ++j) xv[h][j] = x0[kk * LX + j * MS];
        };
#pragma unroll
        for (int i = 0; i < FD - 1; ++i) frag(i * KS, i);
#pragma unroll
        for (int kk = 0; kk < BK; kk += KS) {
            const int h = (kk / KS) % FD;
            if (kk + (FD - 1) * KS < BK) frag(kk + (FD - 1) * KS, (h + FD - 1) % FD);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (MS == 32) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[h][i], xv[h][j], acc[i][j], 0, 0, 0);
                    else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[h][i], xv[h][j], acc[i][j], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // C/D layout: 32x32: col = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5); 16x16: col = lane & 15, row = (lane >> 4) * 4 + r.
    // The residual (or NoiseBlock input) values of the tile are requested together (one by one under their guards they were a memory round trip per
    // row, half of the launch), on the small tile before anything else (the wide one has no registers left for them).
    const bool add = MODE == GEMM_NOISE || MODE == GEMM_RESID || (MODE == GEMM_TAPS && pR);
    const int lde = MODE == GEMM_NOISE ? p.ldx : p.ldy;
    const int row0 = MS == 32 ? 4 * (lane >> 5) : (lane >> 4) * 4;
    const int mw = m0 + wm * TM * MS, mc = min(mw, p.M - 1), mtop = p.M - 1 - mc;       // the wave's first row (scalar), the last row relative to it
    const float* eb = add ? (MODE == GEMM_NOISE ? pX : pR) + ((size_t)b * p.M + mc) * lde : pAT;
    float* yb = pY + ((size_t)b * p.M + mc) * p.ldy;
    float e[TM][TN][NR];
    auto want = [&]() {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * MS + (lane & (MS - 1));
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const int ml = i * MS + (MS == 32 ? (r & 3) + 8 * (r >> 2) : r) + row0;
                    e[i][j][r] = add ? *at(eb, 4 * ((OFF)(IN ? ml : min(ml, mtop)) * lde + (IN ? n : min(n, p.N - 1)))) : 0.0f;
                }
        }
    };
    if constexpr (PRE) want();
    [[maybe_unused]] acc_t tot[QUARTERS ? TM : 1][QUARTERS ? TN : 1];
    [[maybe_unused]] int quarter = 1;
    [[maybe_unused]] auto close_quarter = [&]() {                        // (0 + p0 is p0: a sum that starts at 0 is never -0)
#pragma unroll
        for (int i = 0; i < (QUARTERS ? TM : 0); ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < NR; ++r) { tot[i][j][r] += acc[i][j][r]; acc[i][j][r] = 0.0f; }
    };
    if constexpr (QUARTERS) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) tot[i][j] = acc[i][j];
    }
    // chunk c sits in LDS buffer c & 1; registers hold chunks c + 1 .. c + PF (slot = chunk % PF)
#pragma unroll
    for (int i = 0; i < PF; ++i) load(i, i);
    put(0, 0, 0);
    load(PF, 0);
    __syncthreads();
    // (straight-line groups of PF chunks: a branch around the loads would wait for every load in flight at its join)
    static_assert(PF % 2 == 0, "the LDS buffer of a chunk is its parity inside the group");
    for (int c0 = 0; c0 < nchunks; c0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int slot = (u + 1) % PF;
            put(c0 + u + 1, slot, (u + 1) & 1);
            load(c0 + u + 1 + PF, slot);
            if constexpr (QUARTERS) {
                if (quarter < 4 && (c0 + u) * (BK / 16) == codec_quarter(units, quarter)) { close_quarter(); ++quarter; }
            }
            if (c0 + u < nchunks) math(u & 1);
            __syncthreads();
        }
    }
    if constexpr (QUARTERS) {
        close_quarter();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = tot[i][j];
    }
    if constexpr (!PRE) want();
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + (wn * TN + j) * MS + (lane & (MS - 1));
        const bool nok = IN || n < p.N;
        float nz = 0.0f;
        if (MODE == GEMM_NOISE && nok) {        // explicit tensor, or the documented generator
            if (p.noise) nz = p.noise[(size_t)b * p.N + n];
            else if (p.noise_rng) nz = codec_noise_value(p.noise_key, (uint64_t)(p.row_offset + (p.row_ids ? p.row_ids[b] : b)), n);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float bm[NR];
#pragma unroll
            for (int r = 0; r < NR; ++r) bm[r] = pbias ? pbias[mc + min(i * MS + (MS == 32 ? (r & 3) + 8 * (r >> 2) : r) + row0, mtop)] : 0.0f;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int ml = i * MS + (MS == 32 ? (r & 3) + 8 * (r >> 2) : r) + row0;
                float v = acc[i][j][r] + bm[r];
                if (MODE == GEMM_GELU) v = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));      // exact-erf GELU (VocosBackbone.swift:89)
                if (MODE == GEMM_RESID || MODE == GEMM_TAPS) {
                    if (pscale) v *= pscale[min(mc + ml, p.M - 1)];                                 // ConvNeXt layer scale gamma (VocosBackbone.swift:92-95)
                    if (add) v = e[i][j][r] + v;                                                    // Layers.swift:230
                }
                if (MODE == GEMM_NOISE) v = e[i][j][r] + nz * v;                                    // Layers.swift:276-277
                if (IN || (nok && ml <= mtop && mw < p.M)) *const_cast<float*>(at(yb, 4 * ((OFF)ml * p.ldy + n))) = v;
            }
        }
    }
}
template <int MODE, bool SNAKE, int MS, int WM, int WN, int TM, int TN, int BK, int PF, typename OFF, bool QUARTERS>
__global__ void __launch_bounds__(256, MS == 32 && sizeof(OFF) == 4 ? 3 : 1) k_codec_gemm(GemmParams p, F32Tiles q) {
    constexpr int BM = WM * TM * MS, BN = WN * TN * MS, LA = MS == 32 ? BM : BM + 16, LX = MS == 32 ? BN : BN + 16;
    __shared__ __attribute__((aligned(16))) float As[2 * BK * LA];
    __shared__ __attribute__((aligned(16))) float Xs[2 * BK * LX];
    const int grp = blockIdx.x >> 3, ntile = (blockIdx.x & 7) * q.npx + grp / q.mt, mtile = grp % q.mt, b = blockIdx.y;
    if (ntile >= q.nt) return;
    const int n0 = ntile * BN, m0 = mtile * BM, Cin = MODE == GEMM_TAPS ? p.Cin : p.K;
    const int lo = MODE == GEMM_TAPS ? n0 - p.pad : n0, hi = MODE == GEMM_TAPS ? n0 + BN + (q.taps - 1) * p.dil - p.pad : n0 + BN;
    const bool in = (p.M & 3) == 0 && (Cin & 15) == 0 && (Cin / 16 * q.taps) % (BK / 16) == 0 && ((uintptr_t)p.AT & 15) == 0 && m0 + BM <= p.M && n0 + BN <= p.N &&
                    lo >= p.x_lo && hi <= p.Tin;
    if (in) codec_gemm_tile<MODE, SNAKE, MS, WM, WN, TM, TN, BK, PF, true, OFF, QUARTERS>(p, q.taps, n0, m0, b, As, Xs, p.X, p.R, p.Y, p.bias, p.scale, p.AT);
    else codec_gemm_tile<MODE, SNAKE, MS, WM, WN, TM, TN, BK, PF, false, OFF, QUARTERS>(p, q.taps, n0, m0, b, As, Xs, p.X, p.R, p.Y, p.bias, p.scale, p.AT);
}

// Convolutions with a long K (codec_quarters), the encoders' strided ones among them.  32 x 16 outputs per block, the four waves take a quarter of the K range each
// and meet once in LDS; no staging, both operands come straight from global memory in fragment order (16 lanes = 64 contiguous bytes), four units in
// flight.  768 rows, K = 9216, 296 columns: 94 us (64 x 128 tiles: 652).
#define CODEC_SPLIT_NY 32768       // column tiles in the y dimension of the grid; more of them in z
__device__ __forceinline__ void codec_gemm_split_body(const GemmParams& p, const float* __restrict__ pX, const float* __restrict__ pR, float* __restrict__ pY,
                                                      const float* __restrict__ pbias, const float* __restrict__ pscale, const float* __restrict__ pAT, int batch) {
    constexpr int KW = 4;
    __shared__ float red[KW][32][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.x * 32, b = blockIdx.z % batch, n0 = (blockIdx.z / batch * CODEC_SPLIT_NY + blockIdx.y) * 16;
    if (n0 >= p.N) return;
    const int Cin = p.Cin, T = p.taps;
    const int units = (Cin + 15) / 16 * T, u0 = codec_quarter(units, wave), u1 = codec_quarter(units, wave + 1);
    const float* Xb = pX + (size_t)b * Cin * p.ldx;
    const int kl = lane >> 4, nl = lane & 15;
    const int ma = min(m0 + nl, p.M - 1), mb = min(m0 + 16 + nl, p.M - 1);       // (rows past M are computed and not stored)
    f32x4_t acc[2] = {(f32x4_t){0.f, 0.f, 0.f, 0.f}, (f32x4_t){0.f, 0.f, 0.f, 0.f}};
    struct Unit { float a[4], c[4], x[4]; };
    auto load = [&](Unit& f, int u) {
        u = min(u, units - 1);
        const int cc = u / T, tap = u - cc * T;
        const int n = min(max(n0 + nl + tap * p.dil - p.pad, p.x_lo), p.Tin - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = min(cc * 16 + i * 4 + kl, Cin - 1);
            const float* arow = pAT + (size_t)(tap * Cin + ch) * p.M;
            f.a[i] = arow[ma];
            f.c[i] = arow[mb];
            f.x[i] = Xb[(size_t)ch * p.ldx + n];
        }
    };
    auto math = [&](Unit& f, int u) {
        const int cc = u / T, tap = u - cc * T;
        const int n = n0 + nl + tap * p.dil - p.pad;
        const bool nok = n >= p.x_lo && n < p.Tin;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = cc * 16 + i * 4 + kl;
            float x = f.x[i];
            x = nok && ch < Cin ? x : 0.0f;
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ch < Cin ? f.a[i] : 0.0f, x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ch < Cin ? f.c[i] : 0.0f, x, acc[1], 0, 0, 0);
        }
    };
    Unit f[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) load(f[i], u0 + i);
    for (int u = u0; u < u1; u += 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (u + i < u1) math(f[i], u + i);
            load(f[i], u + 4 + i);
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][t * 16 + kl * 4 + r][nl] = acc[t][r];
    __syncthreads();
    for (int i = tid; i < 32 * 16; i += 256) {
        const int m = m0 + (i >> 4), n = n0 + (i & 15);
        if (m >= p.M || n >= p.N) continue;
        float v = red[0][i >> 4][i & 15];
#pragma unroll
        for (int w = 1; w < KW; ++w) v += red[w][i >> 4][i & 15];
        const size_t o = ((size_t)b * p.M + m) * p.ldy + n;
        if (pbias) v += pbias[m];
        if (pR) {
            if (pscale) v *= pscale[m];
            v = pR[o] + v;
        }
        pY[o] = v;
    }
}
__global__ void __launch_bounds__(256) k_codec_gemm_split(GemmParams p, int batch) { codec_gemm_split_body(p, p.X, p.R, p.Y, p.bias, p.scale, p.AT, batch); }

bool codec_quarters(const GemmParams& p) { return p.K >= 1024; }

template <int MODE, bool SNAKE>
static void launch_f32(const GemmParams& p, int batch, hipStream_t s) {
    // The widest tile that still gives two blocks per compute unit; below that the shape is bound by latency, and the smallest tile has the
    // shortest chain and the most loads in flight.  (Bits do not depend on the choice.)
    auto blocks = [&](int bm, int bn) { return (long)cdiv(p.M, bm) * cdiv(p.N, bn) * batch; };
    auto go = [&](auto kernel, int bm, int bn) {
        F32Tiles q{cdiv(p.N, bn), cdiv(p.M, bm), cdiv(cdiv(p.N, bn), 8), MODE == GEMM_TAPS ? p.taps : 1};
        hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * q.npx * q.mt), batch), dim3(256), 0, s, p, q);
    };
    // A wave's 64 rows lie within 2^32 bytes up to 2^24 samples a row (699 s at 24 kHz); longer ones take 64-bit offsets.
    const bool near = std::max(p.ldx, p.ldy) <= 1 << 24;
    if constexpr (MODE == GEMM_TAPS) {
        if (codec_quarters(p)) {
            // The same bits in all of them.  The tiles where their rows are (nearly) full and their blocks come near to filling the chip once.  us, tiles / split form:
            // 512 rows, K = 3840, 8000 / 9600 / 12000 columns (500 / 600 / 752 blocks) 439 / 500, 541 / 591, 545 / 744; 1024 rows, K = 12288, 5000 columns (632) 1715 /
            // 1937, 1500 columns (192) 1033 / 601; 384 rows, K = 4608, 8000 columns (375) 528 / 450; 64 rows, K = 1536, 60000 columns (469) 187 / 201, 20000 columns
            // 73 / 72; rows three quarters full: 192 rows, K = 1152, 60000 columns (1876) 490 / 442; 48 rows, K = 1536, 100000 columns (782) 370 / 326
            const bool narrow = p.M <= 64;
            if (near && 8 * p.M >= 7 * (narrow ? 64 : cdiv(p.M, 128) * 128) && blocks(narrow ? 64 : 128, narrow ? 128 : 64) >= 448) {
                if (narrow) go(k_codec_gemm<MODE, SNAKE, 32, 1, 4, 2, 1, 16, 2, uint32_t, true>, 64, 128);
                else go(k_codec_gemm<MODE, SNAKE, 32, 2, 2, 2, 1, 16, 2, uint32_t, true>, 128, 64);
            } else {
                const int nt = cdiv(p.N, 16);
                hipLaunchKernelGGL(k_codec_gemm_split, dim3(cdiv(p.M, 32), std::min(nt, CODEC_SPLIT_NY), batch * cdiv(nt, CODEC_SPLIT_NY)), dim3(256), 0, s, p, batch);
            }
            return;
        }
    }
    if (!near) go(k_codec_gemm<MODE, SNAKE, 32, 1, 4, 2, 1, 16, 2, uint64_t, false>, 64, 128);
    else if (p.M <= 64 && blocks(64, 128) >= 512) go(k_codec_gemm<MODE, SNAKE, 32, 1, 4, 2, 1, 16, 2, uint32_t, false>, 64, 128);
    else if (p.M > 64 && blocks(128, 64) >= 512) go(k_codec_gemm<MODE, SNAKE, 32, 2, 2, 2, 1, 16, 2, uint32_t, false>, 128, 64);
    else go(k_codec_gemm<MODE, SNAKE, 16, 2, 2, 1, 1, 64, 4, uint32_t, false>, 32, 32);
}

void launch_gemm_f32(int mode, bool snake, const GemmParams& p, int batch, hipStream_t s) {
    MIS_REQUIRE(mode != GEMM_CONVT && p.M >= 1 && p.N >= 1 && (mode != GEMM_TAPS || (!snake && p.taps >= 1)), MIS_ERR_GENERATION_FAILED, "codec GEMM: bad mode");
    auto run = [&](auto m, auto sn) { launch_f32<decltype(m)::value, decltype(sn)::value>(p, batch, s); };
    const auto off = std::false_type{};
    if (mode == GEMM_PLAIN) run(std::integral_constant<int, GEMM_PLAIN>{}, off);
    else if (mode == GEMM_GELU) run(std::integral_constant<int, GEMM_GELU>{}, off);
    else if (mode == GEMM_RESID && snake) run(std::integral_constant<int, GEMM_RESID>{}, std::true_type{});
    else if (mode == GEMM_RESID) run(std::integral_constant<int, GEMM_RESID>{}, off);
    else if (mode == GEMM_NOISE) run(std::integral_constant<int, GEMM_NOISE>{}, off);
    else run(std::integral_constant<int, GEMM_TAPS>{}, off);
}
