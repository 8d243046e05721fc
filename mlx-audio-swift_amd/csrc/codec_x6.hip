// codec_x6.hip - f32 contractions of the codecs on the bf16 matrix pipe, at f32 accuracy.
//
// Every f32 operand is written EXACTLY as three bfloat16, x = h + m + l, each the nearest to what is left (3 x 8 significant bits, signs absorb the carry),
// and a product becomes the six bf16 MFMAs whose weight is above 2^-24: wh.xh + wh.xm + wm.xh + wm.xm + wh.xl + wl.xh (dropped: wm.xl + wl.xm + wl.xl,
// <= 2^-25 of the product).  One 16-deep step is 6 x 32 cycles instead of 8 x 64 of v_mfma_f32_32x32x2_f32.  Error against 64 bits (2-norm over 2-norm,
// this kernel / the exact-f32 one; K = 96, 128, 192; operands normal): 1.38e-7 / 1.77e-7, 1.65e-7 / 2.06e-7, 2.04e-7 / 2.49e-7; all of one sign: 1.14 / 1.44,
// 1.29 / 1.60, 1.64 / 2.05; normal times exp(2 normal): 1.25 / 1.93, 1.42 / 2.00, 1.84 / 2.45: lower each time (6 roundings of the sum per 16 products, not 16).
// Infinities and values past the largest bfloat16: k_x6_gemm and the encoder's units take the outputs they reach again in f32, k_x6_convt (whose Snake may be the identity) clamps the first
// plane.  Behind a Snake that is none, an argument past 1e20 is infinite or NaN in any arithmetic.  (An infinite WEIGHT of the decoder's units or the transposed
// convolution gives NaN where the f32 kernels give an infinity or NaN.)
//
//   k_x6_pack_w   A^T f32 -> the three planes as MFMA-A fragments (once per weight matrix, kept in the model's CodecPack)
//   k_pw_x6       the fused unit tails of snac.hip (k_pw_fused, which stays for 64 channels without taps and for MIS_CODEC_EXACT_F32=1) and its encoder's units of 48 and 96
//   k_x6_gemm     1x1 and k-tap contractions (codec_f32.hip keeps the rest)
//   k_x6_convt    transposed convolutions of stride 2 and at most 64 rows
#include "common.h"
#include "codec_kernels.h"

#include <algorithm>
#include <type_traits>
#include <utility>


#define X6_MAX 3.38953138925153547590470800371487866880e+38f      // the largest bfloat16
// x = h + m + l exactly (three bfloat16, each the nearest to what is left): eight values of consecutive channels -> one 16-byte piece per plane.
// CLAMP: the first plane of a value past the largest bfloat16 is that one, not infinity; the rest still fits the other two
template <bool CLAMP>
__device__ __forceinline__ void x6_split(const float (&v)[8], uint4& h, uint4& m, uint4& l) {
    uint32_t o[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const float ca = q || !CLAMP ? a : __builtin_amdgcn_fmed3f(a, -X6_MAX, X6_MAX), cb = q || !CLAMP ? b : __builtin_amdgcn_fmed3f(b, -X6_MAX, X6_MAX);
            const uint32_t ab = (uint32_t)f32_to_bf16(ca) | ((uint32_t)f32_to_bf16(cb) << 16);
            o[q][i] = ab;
            a -= __uint_as_float(ab << 16);
            b -= __uint_as_float(ab & 0xffff0000u);
        }
    }
    h = make_uint4(o[0][0], o[0][1], o[0][2], o[0][3]);
    m = make_uint4(o[1][0], o[1][1], o[1][2], o[1][3]);
    l = make_uint4(o[2][0], o[2][1], o[2][2], o[2][3]);
}

// A^T f32 [ntaps][Cin][M] -> fragments of v_mfma_f32_32x32x16_bf16: [Cin / 16][tap][MT32][plane][64 lanes][8]
__global__ void k_x6_pack_w(const float* __restrict__ AT, uint16_t* __restrict__ wp, int ntaps, int Cin, int M, int MT32, int KS) {
    const size_t total = (size_t)ntaps * KS * MT32 * 512;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const int j = (int)(e & 7), lane = (int)((e >> 3) & 63);
        size_t r = e >> 9;
        const int mt = (int)(r % MT32); r /= MT32;
        const int tap = (int)(r % ntaps);
        const int ks = (int)(r / ntaps);
        const int m = mt * 32 + (lane & 31), c = ks * 16 + (lane >> 5) * 8 + j;
        float v = (m < M && c < Cin) ? AT[((size_t)tap * Cin + c) * M + m] : 0.0f;
        const size_t o = (e >> 9) * 1536 + (size_t)lane * 8 + j;
        for (int q = 0; q < 3; ++q) {
            const uint16_t h = f32_to_bf16(q ? v : __builtin_amdgcn_fmed3f(v, -X6_MAX, X6_MAX));
            wp[o + q * 512] = h;
            v -= bf16_to_f32(h);
        }
    }
}

const CodecPack::X6& CodecPack::get_x6(const float* at, int ntaps, int Cin, int M, hipStream_t s) {
    for (auto& e : x6)
        if (e.at == at && e.ntaps == ntaps && e.Cin == Cin && e.M == M) return e;
    X6 e{};
    e.at = at; e.ntaps = ntaps; e.Cin = Cin; e.M = M;
    e.KS = (Cin + 15) / 16;
    e.MT32 = (M + 31) / 32;
    const size_t n = (size_t)ntaps * e.KS * e.MT32 * 1536;
    HIP_CHECK(hipMalloc((void**)&e.wp, n * sizeof(uint16_t)));
    hipLaunchKernelGGL(k_x6_pack_w, dim3((unsigned)std::min<size_t>((n / 3 + 255) / 256, 8192)), dim3(256), 0, s, at, e.wp, ntaps, Cin, M, e.MT32, e.KS);
    x6.push_back(e);
    return x6.back();
}

// ---- fused residual unit tails --------------------------------------------------------------------------------------------------------
// The kernels of k_pw_fused (snac.hip), chunk by chunk: DW: x with its dilation halo -> Snake -> LDS -> seven taps, bias, Snake; else Snake alone; then eight
// channels of a column per thread are split and written as one 16-byte piece per plane, [plane][channel / 8][column], which is the MFMA-B fragment.
// What bounds it: k_pw_fused<128, DW> took 1.05 ms without its MFMAs (4.8 GB of loads and stores, 32 rows of 98304 columns) and 1.75 ms with: the f32
// matrix time adds to the memory time.  Six bf16 products take 0.25 instead of 0.68 ms of it: 1.95 -> 1.44 ms.
typedef uint32_t x6_u4 __attribute__((ext_vector_type(4)));
struct PwScalars { int T, ldx, ldr, ldy, nbx, per, tiles; };
// LDS alone: __syncthreads() would wait for the next chunk's samples and weights as well
__device__ __forceinline__ void pw_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
template <int C, int DIL, int KC, int NT, bool PF, bool OUT>
__device__ __forceinline__ void pw_x6_body(const float* __restrict__ pX, const float* __restrict__ pR, float* __restrict__ pY,
                                           const float* __restrict__ pw7, const float* __restrict__ pb1, const float* __restrict__ pa1,
                                           const float* __restrict__ pra1, const float* __restrict__ pa2, const float* __restrict__ pra2,
                                           const uint16_t* __restrict__ pwp, const float* __restrict__ pAT, const float* __restrict__ pb2, const PwScalars p, const CodecPlanes po,
                                           const float* __restrict__ poa, const float* __restrict__ pora, uint16_t* __restrict__ pout) {
    constexpr int KG = KC / 8, MT = (C + 31) / 32, APC = KC / 16 * MT * 192;       // channel groups, row tiles, 16-byte pieces of weights per chunk
    constexpr bool DW = DIL > 0;
    constexpr int XR = KC / 4, NS = NT / 64, GS = KG * NS / 4;                      // rows of x, strips of columns, (group, strip) pairs per wave
    // The dilation is a constant: as many columns are staged as it needs.  The halo of a wave's rows comes one row behind the other, 64 values at a time, each with its Snake's
    // parameters; in chunks of 16 at most HR rows a load, whose parameters are scalar then - 16 registers less, a block more a compute unit (us, without / with: 64 channels,
    // 49152 blocks, dilation 3 1180 / 1100, 9 1212 / 1097; 48, 1181 blocks, 9 28.4 / 22.8; 96, 592 blocks, 9 36.8 / 34.8, 3776 blocks 182 / 158; 128, 24576 blocks, 9 1440 / 1395;
    // but 3 1400 / 1500, 96 channels 3 32.4 / 33.6; chunks of 32, 128 channels in 64 columns: 3 19.7 / 21.2, 9 17.1 / 21.8; 64 channels 3 12.7 / 13.4)
    constexpr int HALO = 3 * DIL, XS = NT + 2 * HALO + 2, HR = KC != 16 ? 0 : DIL == 9 ? 1 : DIL == 3 && C <= 64 ? 2 : 0, HP = HR ? XR / (HR ? HR : 1) : (XR * 2 * HALO + 63) / 64;
    static_assert(HR * 2 * HALO <= 64 && (!HR || XR % HR == 0), "a wave holds the halo of HR rows");
    __shared__ float xs[DW ? KC : 1][DW ? XS : 1];
    __shared__ uint4 sm[3 * KG * NT + APC];
    uint4 (&ts)[3][KG][NT] = *reinterpret_cast<uint4 (*)[3][KG][NT]>(sm);
    x6_u4 (&As)[APC] = *reinterpret_cast<x6_u4 (*)[APC]>(sm + 3 * KG * NT);
    // Units of 48 and 96 channels (the encoder's) take the place of k_x6_gemm in long rows only, those of 64 (the decoder's) of an f32 kernel: a lane that sees a sum which is not
    // finite takes its rows again as those do
    constexpr bool RETAKE = DW && C <= 96;
    constexpr bool SQ = C == 128 || NT == 64;             // 2 x 2 waves of half the rows and half the columns; else every wave: all C rows x 32 columns
    constexpr int MTW = SQ ? MT / 2 : MT, NTW = SQ ? NT / 64 : 1;
    static_assert(SQ ? MT % 2 == 0 : NT == 128, "2 x 2 waves, or four of 32 columns");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (an XCD takes a contiguous range of blocks: a neighbour's halo and the other half of a line are in its L2)
    const int tileid = (blockIdx.x & 7) * p.per + (blockIdx.x >> 3);
    if (tileid >= p.tiles) return;
    const int b = tileid / p.nbx, n0 = (tileid - b * p.nbx) * NT;
    const int wr = SQ ? (wave >> 1) * MTW : 0;              // first row tile / first column of the wave's tile
    const int wc = SQ ? (wave & 1) * (NT / 2) : wave * 32;
    const float* xb = pX + (size_t)b * C * p.ldx;
    const int T = p.T;
    f32x16_t acc[MTW][NTW];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    x6_u4 wv[(APC + 255) / 256];
    float vx[DW ? XR : GS][DW ? NS : 8], vh[DW ? HP : 1], ah[DW && !HR ? HP : 1], rah[DW && !HR ? HP : 1];
    const auto halo = [&](int h, int& r, int& j) {                         // the lane's value of load h of the halo: its row, its column of xs; false: none
        const int i = HR ? (HR == 2 && lane >= 2 * HALO) : (h * 64 + lane) / max(2 * HALO, 1);
        j = min((HR ? 0 : h * 64) + lane - i * 2 * HALO, max(2 * HALO - 1, 0));
        j += j < HALO ? 0 : NT;
        r = min(h * HR + i, XR - 1);
        return HR ? lane < HR * 2 * HALO : h * 64 + lane < XR * 2 * HALO;
    };
    auto fetch = [&](int c0) {
        const x6_u4* wsrc = reinterpret_cast<const x6_u4*>(pwp) + (size_t)(c0 / 16) * MT * 192;
#pragma unroll
        for (int i = 0; i < (APC + 255) / 256; ++i) wv[i] = wsrc[min(tid + i * 256, APC - 1)];
        if constexpr (DW) {
#pragma unroll
            for (int r = 0; r < XR; ++r)
#pragma unroll
                for (int sx = 0; sx < NS; ++sx) vx[r][sx] = xb[(size_t)(c0 + wave + 4 * r) * p.ldx + min(n0 + sx * 64 + lane, T - 1)];
#pragma unroll
            for (int h = 0; h < HP; ++h) {
                int r, j;
                halo(h, r, j);
                const int c = c0 + wave + 4 * r;
                vh[h] = xb[(size_t)c * p.ldx + min(max(n0 - HALO + j, 0), T - 1)];
                if constexpr (!HR) { ah[h] = pa1[c]; rah[h] = pra1[c]; }
            }
        } else {
#pragma unroll
            for (int g = 0; g < GS; ++g) {
                const int kg = KC == 32 ? wave : wave >> 1, n = (KC == 32 ? g : wave & 1) * 64 + lane;
#pragma unroll
                for (int j = 0; j < 8; ++j) vx[g][j] = xb[(size_t)(c0 + kg * 8 + j) * p.ldx + min(n0 + n, T - 1)];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (PF) fetch(0);
    for (int c0 = 0; c0 < C; c0 += KC) {
        if constexpr (PF) pw_lds_barrier(); else __syncthreads();          // the previous chunk's MFMAs are done with ts / As
        if (!PF) fetch(c0);
        if (DW) {
#pragma unroll
            for (int r = 0; r < XR; ++r) {
                const int cc = wave + 4 * r, c = c0 + cc;
                const float al = pa1[c], ral = pra1[c];
#pragma unroll
                for (int sx = 0; sx < NS; ++sx) {
                    const int j = sx * 64 + lane;
                    xs[cc][HALO + j] = mis_snake(n0 + j < T ? vx[r][sx] : 0.0f, al, ral);
                }
                __builtin_amdgcn_sched_barrier(0);                          // (a row at a time: the values in flight take the registers)
            }
#pragma unroll
            for (int h = 0; h < HP; ++h) {
                int r, j;
                const bool on = halo(h, r, j);
                const int t = n0 - HALO + j;
                float al = ah[HR ? 0 : h], ral = rah[HR ? 0 : h];
                if constexpr (HR > 0) {
                    const int c = c0 + wave + 4 * HR * h;
                    al = pa1[c]; ral = pra1[c];
                    if constexpr (HR == 2) { const float a1 = pa1[c + 4], ra1 = pra1[c + 4]; if (r & 1) { al = a1; ral = ra1; } }
                }
                const float u = mis_snake(t >= 0 && t < T ? vh[h] : 0.0f, al, ral);
                if (on) xs[wave + 4 * r][j] = u;
            }
        } else {
#pragma unroll
            for (int g = 0; g < GS; ++g) {
                const int kg = KC == 32 ? wave : wave >> 1, n = (KC == 32 ? g : wave & 1) * 64 + lane;
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = mis_snake(vx[g][j], pa2[c0 + kg * 8 + j], pra2[c0 + kg * 8 + j]);
                uint4 h, m, l;
                x6_split<false>(v, h, m, l);
                ts[0][kg][n] = h; ts[1][kg][n] = m; ts[2][kg][n] = l;
            }
        }
#pragma unroll
        for (int i = 0; i < (APC + 255) / 256; ++i)
            if (APC % 256 == 0 || tid + i * 256 < APC) As[tid + i * 256] = wv[i];
        if constexpr (PF) {
            __builtin_amdgcn_sched_barrier(0);
            if (c0 + KC < C) fetch(c0 + KC);                                // (in flight behind this chunk's taps and products)
        }
        if (DW) {
            if constexpr (PF) pw_lds_barrier(); else __syncthreads();
            // depthwise taps + bias + Snake -> eight channels of one column per thread (consecutive lanes read consecutive LDS words)
#pragma unroll
            for (int g = 0; g < GS; ++g) {
                const int kg = KC == 32 ? wave : wave >> 1, n = (KC == 32 ? g : wave & 1) * 64 + lane;
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int cc = kg * 8 + j, c = c0 + cc;
                    float a = 0.0f;
#pragma unroll
                    for (int k = 0; k < 7; ++k) a += pw7[c * 7 + k] * xs[cc][n + k * DIL];
                    v[j] = mis_snake(a + pb1[c], pa2[c], pra2[c]);
                    if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                uint4 h, m, l;
                x6_split<false>(v, h, m, l);
                ts[0][kg][n] = h; ts[1][kg][n] = m; ts[2][kg][n] = l;
            }
        }
        if constexpr (PF) pw_lds_barrier(); else __syncthreads();
#pragma unroll
        for (int ks = 0; ks < KC / 16; ++ks) {
            bf16x8_t bv[NTW][3];
#pragma unroll
            for (int ni = 0; ni < NTW; ++ni)
#pragma unroll
                for (int q = 0; q < 3; ++q) bv[ni][q] = *reinterpret_cast<const bf16x8_t*>(&ts[q][2 * ks + (lane >> 5)][wc + ni * 32 + (lane & 31)]);
            constexpr int MP = NTW == 1 && MTW % 2 == 0 ? 2 : 1;             // row tiles at a time: two accumulators alternate
#pragma unroll
            for (int m0 = 0; m0 < MTW; m0 += MP) {
                bf16x8_t av[MP][3];
#pragma unroll
                for (int mi = 0; mi < MP; ++mi)
#pragma unroll
                    for (int q = 0; q < 3; ++q) av[mi][q] = *reinterpret_cast<const bf16x8_t*>(&As[((ks * MT + wr + m0 + mi) * 3 + q) * 64 + lane]);
                // smallest first: w_l x_h, w_h x_l, w_m x_m, w_m x_h, w_h x_m, w_h x_h
                constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int mi = 0; mi < MP; ++mi)
#pragma unroll
                        for (int ni = 0; ni < NTW; ++ni)
                            acc[m0 + mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi][QA[q]], bv[ni][QB[q]], acc[m0 + mi][ni], 0, 0, 0);
            }
        }
    }
    // epilogue: + bias + residual (C/D layout: col = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5))
    const float* rb = pR + (size_t)b * C * p.ldr;
    float* yb = pY + (size_t)b * C * p.ldy;
    if constexpr (OUT) {                                       // as the operand of the contraction behind, and in f32 where something else reads it; the next tile's residual requested ahead
        static_assert(sizeof(sm) >= 4 * CP_LDS(2) * sizeof(uint16_t), "the staging buffers hold the waves' output tiles");
        uint16_t* st = reinterpret_cast<uint16_t*>(sm) + wave * CP_LDS(2);
        __syncthreads();                                       // (the other waves' products)
        float e[2][16];
        auto want = [&](int t, float (&v)[16]) {
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = rb[(size_t)((wr + t / NTW) * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5)) * p.ldr + min(n0 + wc + t % NTW * 32 + (lane & 31), T - 1)];
        };
        want(0, e[0]);
#pragma unroll
        for (int t = 0; t < MTW * NTW; ++t) {
            const int mi = t / NTW, ni = t % NTW, nb = n0 + wc + ni * 32, n = nb + (lane & 31);
            if (t + 1 < MTW * NTW) want(t + 1, e[(t + 1) & 1]);
#pragma unroll
            for (int r0 = 0; r0 < 16; r0 += 8) {
                const int m0 = (wr + mi) * 32 + 2 * r0 + 4 * (lane >> 5);
                float y[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) y[r] = e[t & 1][r0 + r] + (acc[mi][ni][r0 + r] + pb2[m0 + (r & 3) + 8 * (r >> 2)]);
                if (pY && n < T) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) yb[(size_t)(m0 + (r & 3) + 8 * (r >> 2)) * p.ldy + n] = y[r];
                }
                if (poa) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) { const int m = m0 + (r & 3) + 8 * (r >> 2); y[r] = mis_snake(y[r], poa[m], pora[m]); }
                }
                codec_tile_put<2>(y, st, r0, lane);
            }
            codec_tile_flush<2>(st, pout + (size_t)b * po.Tp * C + (wr + mi) * 32, po.stride, C, lane, [&](int c) {
                const int r = nb + c - po.t_org;
                return nb + c < T && r < po.Tp ? r : -1;
            });
        }
        codec_plane_ends(po, b, T, 0, C, n0 == 0, n0 + NT >= T, tid, 256);
        return;
    }
#pragma unroll
    for (int ni = 0; ni < NTW; ++ni) {
        const int n = n0 + wc + ni * 32 + (lane & 31);
        if (n >= T) continue;
#pragma unroll
        for (int mi = 0; mi < MTW; ++mi) {
            if constexpr (RETAKE) {
                float zero = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; ++r) zero = fmaf(acc[mi][ni][r], 0.0f, zero);
                if (zero != 0.0f) {
#pragma unroll 1
                    for (int r = 0; r < 16; ++r) {
                        const int m = (wr + mi) * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
                        if (m >= C) break;
                        float v = 0.0f;
#pragma unroll 1
                        for (int c = 0; c < C && v == v; ++c) {            // (NaN it stays)
                            float a = 0.0f;
#pragma unroll 1
                            for (int k = 0; k < 7; ++k) {
                                const int t = n + (k - 3) * DIL;
                                a = fmaf(pw7[c * 7 + k], mis_snake(t >= 0 && t < T ? xb[(size_t)c * p.ldx + t] : 0.0f, pa1[c], pra1[c]), a);
                            }
                            v = fmaf(pAT[(size_t)c * C + m], mis_snake(a + pb1[c], pa2[c], pra2[c]), v);
                        }
                        yb[(size_t)m * p.ldy + n] = rb[(size_t)m * p.ldr + n] + (v + pb2[m]);
                    }
                    continue;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = (wr + mi) * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
                if (C % 32 == 0 || m < C) yb[(size_t)m * p.ldy + n] = rb[(size_t)m * p.ldr + n] + (acc[mi][ni][r] + pb2[m]);
            }
        }
    }
}
// Blocks a compute unit: chunks of 32 channels two; chunks of 16 as many as the registers allow without spills (us, three / five: 48 channels, 1181 blocks, dilation 1 28.6 / 23.3;
// 64, 49152 blocks, dilation 1 1169 / 1067; dilation 9 with its halo's parameters in registers spilled at five: 1891)
template <int C, int DIL, int KC, int NT, bool PF, bool OUT>
__global__ void __launch_bounds__(256, KC == 32 ? 2 : DIL ? (C <= 64 ? 5 : C == 96 ? 4 : 3) : OUT && C >= 96 ? 3 : 4) k_pw_x6(PwFusedParams p, const uint16_t* wp, CodecPlanes o) {
    pw_x6_body<C, DIL, KC, NT, PF, OUT>(p.X, p.R, p.Y, p.w7, p.b1, p.a1, p.ra1, p.a2, p.ra2, wp, p.AT, p.b2, PwScalars{p.T, p.ldx, p.ldr, p.ldy, p.nbx, p.per, p.tiles}, o, o.alpha, o.ralpha, o.p);
}

// 128 channels, at most 256 blocks of 128 columns (a compute unit each, one serial chain of chunks): 64 columns per block.  96 blocks: 28 -> 22 us;
// 192 and 248: 23 and 25 (384 of 128 columns: 34).
// Chunk depth (the same bits): 32 channels need half the barriers, 16 let three or four blocks (not two, C = 96: three) share a compute unit.  32 while its
// blocks are all resident at once, else 16 (us, chunks of 32 / 16): 128 channels 96 blocks 28 / 33, 384: 34 / 38, 576: 61 / 45, 24576: 1584 / 1430;
// 96 channels 626 blocks: 26.5 / 28.3, 4004: 162 / 150 (with taps 16: 592 blocks, two rounds of 32).  192 channels hold 96 accumulators either way: 313 blocks 36.6 / 52.4, 2004: 193 / 215, always 32;
// up to 512 blocks 64 columns (half the conversions and accumulators per thread, three blocks a compute unit): 313 blocks with planes out 50 -> 42.
// PF, the next chunk's samples and weights requested behind this one's staging (us, without / with): 192 channels 42.4 / 40.1 and 259 / 246, 96 without taps 24.0 / 22.8 and 145.7 / 138,
// 128 in 64 columns 22 / 16-20; chunks of 16 with taps are slower for it (64 channels, 49152 blocks: 1169 / 1364-1522; 48, 7500: 149 / 179-202), 128 in blocks of 128 columns keep a
// third block a compute unit instead (24576 blocks 1400 / 1650).
template <int C, int DIL>
static void launch_x6(const PwFusedParams& p, const uint16_t* wp, int batch, hipStream_t s) {
#define X6_GO(KC, NT, PF) do { \
        PwFusedParams f = p; \
        f.nbx = (p.T + NT - 1) / NT; f.tiles = f.nbx * batch; f.per = (f.tiles + 7) / 8; \
        const dim3 g(8 * f.per); \
        if (!DIL && p.out) hipLaunchKernelGGL((k_pw_x6<C, DIL, KC, NT, PF, !DIL>), g, dim3(256), 0, s, f, wp, *p.out); \
        else hipLaunchKernelGGL((k_pw_x6<C, DIL, KC, NT, PF, false>), g, dim3(256), 0, s, f, wp, CodecPlanes{}); \
        return; } while (0)
    const int64_t blocks = (int64_t)((p.T + 127) / 128) * batch;
    if constexpr (C == 48) X6_GO(16, 128, false);
    else if constexpr (C == 192) {
        if (blocks <= 512) X6_GO(32, 64, true);
        X6_GO(32, 128, true);
    } else {
        if constexpr (C == 128) {
            if (blocks <= 256) X6_GO(32, 64, true);
        }
        if (blocks > (C == 96 && !DIL ? 768 : 512)) X6_GO(16, 128, DIL == 0 && C != 128);
        X6_GO(32, 128, C != 128);
    }
#undef X6_GO
}

// 64 channels with taps: one form for every length, as a row's bits must not change with it.  us, k_pw_fused / here, dilations of 1, 3 and 9: 192 blocks 17.2 / 13.5 12.8 13.4,
// 288: 19.0 / 15.1 14.9 15.6, 768: 26.1 / 23.8 23.8 23.8, 49152: 1122 / 1067 1090 1083.  Without taps (HBM-bound there: twice the columns per product) they stay on k_pw_fused.
bool launch_pw_x6(int C, bool dw, const PwFusedParams& p, CodecPack* pack, int batch, hipStream_t s) {
    if (!pack) pack = codec_x6_scope();
    if (!pack || codec_exact_f32() || (dw && p.dil != 1 && p.dil != 3 && p.dil != 9) || !(dw ? C == 48 || C == 64 || C == 96 || C == 128 : (C == 96 || C == 128 || C == 192))) return false;
    MIS_REQUIRE(!p.out || (!dw && p.out->n == 2 && p.out->Cp == C), MIS_ERR_GENERATION_FAILED, "codec unit: %d rows for %d planes of %d channels", C, p.out->n, p.out->Cp);
    const uint16_t* wp = pack->get_x6(p.AT, 1, C, C, s).wp;
    auto taps = [&](auto c) {
        constexpr int W = decltype(c)::value;
        if (p.dil == 1) launch_x6<W, 1>(p, wp, batch, s);
        else if (p.dil == 3) launch_x6<W, 3>(p, wp, batch, s);
        else launch_x6<W, 9>(p, wp, batch, s);
    };
    if (dw && C == 48) taps(std::integral_constant<int, 48>{});
    else if (dw && C == 64) taps(std::integral_constant<int, 64>{});
    else if (dw && C == 96) taps(std::integral_constant<int, 96>{});
    else if (dw) taps(std::integral_constant<int, 128>{});
    else if (C == 96) launch_x6<96, 0>(p, wp, batch, s);
    else if (C == 128) launch_x6<128, 0>(p, wp, batch, s);
    else launch_x6<192, 0>(p, wp, batch, s);
    return true;
}

// ---- 1x1 and k-tap contractions -----------------------------------------------------------------------------------------------------------
// A wave owns 32 columns and MTW row tiles: it reads its eight channels of a column per lane straight from memory, converts them once and multiplies them
// with all its rows, so the activations need neither LDS nor a barrier.  WIDE: the four waves of a block share the weights, staged in LDS two chunks deep;
// else (few blocks) one row tile per block, weights straight into registers.  k order: 16 channels, within them the taps, six products each.
// Bound (256 x 256 with residual, 32 x 24576 columns): 2.4 GB = 0.49 ms of the 0.85; the products' 0.53 ms run half behind it.
struct X6Gemm {
    GemmParams g;
    int mode, ntaps, nsteps, MT32;        // steps of 16 channels of one tap
    int nbx, my, per, tiles;              // column tiles, row tiles, tiles per XCD, all tiles
    CodecPlanes out;
};
// QUARTERS (codec_quarters: K >= 1024): four partial sums.  The narrow form's four waves then share 32 columns and take a quarter of the steps each; the wide one
// adds its accumulators to the total at the same steps, so a row's bits do not depend on which of them its length selects.
template <class F, int... I>
__device__ __forceinline__ void x6_each(F& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int MTW, bool SNAKE, bool TAPS, bool WIDE, bool QUARTERS, bool OUT>
__device__ __forceinline__ void x6_gemm_body(const X6Gemm& P, const float* __restrict__ pX, const float* __restrict__ pR, float* __restrict__ pY,
                                             const float* __restrict__ pbias, const float* __restrict__ pscale, const float* __restrict__ pnoise,
                                             const float* __restrict__ pa, const float* __restrict__ pra, const float* __restrict__ pAT,
                                             const uint16_t* __restrict__ pwp, const float* __restrict__ poa, const float* __restrict__ pora, uint16_t* __restrict__ pout) {
    constexpr bool TIGHT = MTW == 8 || (MTW == 4 && QUARTERS), KSPLIT = QUARTERS && !WIDE;
    constexpr int PF = TIGHT ? 2 : 4, SPB = TIGHT ? 1 : 2;                  // steps of X (narrow: of weights too) in flight; steps per staged chunk of weights
    constexpr int NA = (SPB * MTW * 192 + 255) / 256, APC = SPB * MTW * 192;
    __shared__ x6_u4 As[WIDE ? 2 : 1][WIDE ? APC : 1];
    __shared__ float red[KSPLIT ? 4 : 1][KSPLIT ? 16 : 1][KSPLIT ? 64 : 1];
    __shared__ __attribute__((aligned(16))) uint16_t tiles[OUT ? 4 : 1][OUT ? CP_LDS(2) : 1];
    extern __shared__ float x6_ab[];                                        // SNAKE: alpha [K], 1 / alpha [K]
    const GemmParams& p = P.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kh = lane >> 5;
    const int tileid = (blockIdx.x & 7) * P.per + (blockIdx.x >> 3);
    if (tileid >= P.tiles) return;
    const int by = tileid % P.my, bxb = tileid / P.my, bx = bxb % P.nbx, b = bxb / P.nbx;
    const int n = (KSPLIT ? bx * 32 : bx * 128 + wave * 32) + (lane & 31), nc = min(n, p.N - 1);
    const int lo = KSPLIT ? codec_quarter(P.nsteps, wave) : 0, hi = KSPLIT ? codec_quarter(P.nsteps, wave + 1) : P.nsteps;      // this wave's steps
    const int mt0 = by * MTW, Kx = TAPS ? p.Cin : p.K;
    if constexpr (SNAKE) {
        for (int i = tid; i < Kx; i += 256) { x6_ab[i] = pa[i]; x6_ab[Kx + i] = pra[i]; }
        __syncthreads();
    }
    if (!WIDE && !KSPLIT && bx * 128 + wave * 32 >= p.N) return;            // (no barrier below)
    const float* xb = pX + ((size_t)b * Kx + kh * 8) * p.ldx;
    const x6_u4* wsrc = reinterpret_cast<const x6_u4*>(pwp) + (size_t)mt0 * 192;
    const size_t wstep = (size_t)P.MT32 * 192;
    const int mtop = (P.MT32 - mt0) * 192 - 1;                              // last piece of this block's rows within a step
    float v[PF][8];
    bool ok[PF];
    x6_u4 aw[WIDE ? 1 : PF][MTW][3];
    int fs = lo, ftap = KSPLIT ? lo % P.ntaps : 0;                          // next step to request
    const float* fx = xb + (KSPLIT ? (size_t)(lo / P.ntaps) * 16 * p.ldx : 0);
    auto fetch = [&](int slot) {
        const int t = TAPS ? nc - p.pad + ftap * p.dil : nc;
        ok[slot] = !TAPS || (t >= p.x_lo && t < p.Tin);
        const float* r = fx + (TAPS ? min(max(t, p.x_lo), p.Tin - 1) : t);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[slot][j] = r[(size_t)j * p.ldx];
        if constexpr (!WIDE) {
#pragma unroll
            for (int mi = 0; mi < MTW; ++mi)
#pragma unroll
                for (int q = 0; q < 3; ++q) aw[slot][mi][q] = wsrc[(size_t)fs * wstep + min((mi * 3 + q) * 64 + lane, mtop)];
        }
        if (fs + 1 < hi) {                                                  // (past the end: the last step again)
            ++fs;
            if (!TAPS || ++ftap == P.ntaps) { ftap = 0; fx += (size_t)16 * p.ldx; }
        }
    };
    x6_u4 wv[NA];
    auto loadA = [&](int c) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = min(tid + i * 256, APC - 1), st = e / (MTW * 192), o = e - st * (MTW * 192);
            wv[i] = wsrc[(size_t)min(c * SPB + st, P.nsteps - 1) * wstep + min(o, mtop)];
        }
    };
    auto putA = [&](int h) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (APC % 256 == 0 || tid + i * 256 < APC) As[h][tid + i * 256] = wv[i];
    };
        // Epilogue values (the modes of k_codec_gemm; C/D layout: col = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5)): a tile's bias, scale and residual or
    // NoiseBlock input, requested together - the narrow form's before its contraction.
    const bool noise = P.mode == GEMM_NOISE, gelu = P.mode == GEMM_GELU;
    const float* eb = noise ? pX + (size_t)b * p.K * p.ldx : (!gelu && pR) ? pR + (size_t)b * p.M * p.ldy : nullptr;
    const int lde = noise ? p.ldx : p.ldy;
    const float* bp = pbias ? pbias : pX;                                   // (loaded either way: a guard per value would be a round trip per value)
    const int btop = pbias ? p.M - 1 : 0;
    float nz = 0.0f;
    if (noise && n < p.N) {
        if (pnoise) nz = pnoise[(size_t)b * p.N + n];
        else if (p.noise_rng) nz = codec_noise_value(p.noise_key, (uint64_t)(p.row_offset + (p.row_ids ? p.row_ids[b] : b)), n);
    }
    constexpr int NR = KSPLIT ? 4 : 16;                                     // rows of a tile that a lane finishes
    float bm[NR], sc[NR], e[NR];
    auto want = [&](int mi, int lane_hi) {
        const int m0 = (mt0 + mi) * 32 + 4 * lane_hi + (KSPLIT ? 8 * wave : 0);
#pragma unroll
        for (int r = 0; r < NR; ++r) bm[r] = bp[min(m0 + (r & 3) + 8 * (r >> 2), btop)];
        if (pscale) {
#pragma unroll
            for (int r = 0; r < NR; ++r) sc[r] = pscale[min(m0 + (r & 3) + 8 * (r >> 2), p.M - 1)];
        }
        if (eb) {
#pragma unroll
            for (int r = 0; r < NR; ++r) e[r] = eb[(size_t)min(m0 + (r & 3) + 8 * (r >> 2), p.M - 1) * lde + nc];
        }
    };
    if constexpr (!WIDE) want(0, kh);
    f32x16_t acc[MTW];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    int ks = 0, tap = 0;                                                    // step being multiplied (SNAKE: its channels)
    bf16x8_t bv[2][3];
    auto convert = [&](int slot, int h2) {
        float x[8];
        [[maybe_unused]] const int kc = min(ks * 16, Kx - 16) + kh * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] = v[slot][j];
            if constexpr (SNAKE) x[j] = mis_snake(x[j], x6_ab[kc + j], x6_ab[Kx + kc + j]);
            if constexpr (TAPS) x[j] = ok[slot] ? x[j] : 0.0f;
        }
        uint4 h, m, l;
        x6_split<false>(x, h, m, l);
        bv[h2][0] = __builtin_bit_cast(bf16x8_t, h); bv[h2][1] = __builtin_bit_cast(bf16x8_t, m); bv[h2][2] = __builtin_bit_cast(bf16x8_t, l);
        if (!TAPS || ++tap == P.ntaps) { tap = 0; ++ks; }
    };
    constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};   // as pw_x6_body
    auto products = [&](int h2, auto frag) {
        constexpr int MP = MTW >= 2 ? 2 : 1;
#pragma unroll
        for (int m0 = 0; m0 < MTW; m0 += MP) {
            bf16x8_t av[MP][3];
#pragma unroll
            for (int mi = 0; mi < MP; ++mi)
#pragma unroll
                for (int q = 0; q < 3; ++q) av[mi][q] = __builtin_bit_cast(bf16x8_t, frag(m0 + mi, q));
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int mi = 0; mi < MP; ++mi) acc[m0 + mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi][QA[q]], bv[h2][QB[q]], acc[m0 + mi], 0, 0, 0);
        }
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) fetch(i);
    // One scheduling region per step: this step's products, the next one's conversion, the request of the step PF ahead.  (With guards between them the
    // conversion waits for the products; without the barrier the scheduler moves the requests to their use.)
    convert(0, 0);
    if constexpr (WIDE) {
        constexpr int CG = PF / SPB;                                        // chunks per straight-line group: PF steps, an even number of chunks
        static_assert(CG % 2 == 0, "the LDS buffer of a chunk is its parity inside the group");
        const int nchunks = (P.nsteps + SPB - 1) / SPB;
        loadA(0);
        putA(0);
        loadA(1);
        __syncthreads();
        f32x16_t tot[QUARTERS ? MTW : 1];
        int quarter = 1;
        [[maybe_unused]] auto close_quarter = [&]() {                       // (0 + p0 is p0: a sum that starts at 0 is never -0)
#pragma unroll
            for (int i = 0; i < MTW; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) { tot[QUARTERS ? i : 0][r] += acc[i][r]; acc[i][r] = 0.0f; }
        };
        if constexpr (QUARTERS) {
#pragma unroll
            for (int i = 0; i < MTW; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) tot[i][r] = 0.0f;
        }
        auto group = [&](int c0, auto whole) {
            if constexpr (QUARTERS) {
                if (quarter < 4 && c0 * SPB == codec_quarter(P.nsteps, quarter)) { close_quarter(); ++quarter; }
            }
#pragma unroll
            for (int u = 0; u < CG; ++u) {
                putA((u + 1) & 1);
                loadA(c0 + u + 2);
#pragma unroll
                for (int st = 0; st < SPB; ++st) {
                    const int slot = u * SPB + st;
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(slot);
                    if (decltype(whole)::value || c0 * SPB + slot < P.nsteps) products(slot & 1, [&](int mi, int q) { return As[u & 1][(st * MTW + mi) * 192 + q * 64 + lane]; });
                    convert((slot + 1) % PF, (slot + 1) & 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                __syncthreads();
            }
        };
        int c0 = 0;
        for (; (c0 + CG) * SPB <= P.nsteps; c0 += CG) group(c0, std::true_type{});
        if (c0 < nchunks) group(c0, std::false_type{});
        if constexpr (QUARTERS) {
            close_quarter();
#pragma unroll
            for (int i = 0; i < MTW; ++i) acc[i] = tot[i];
        }
    } else {
        auto group = [&](int s0, auto whole) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                x6_u4 a[MTW][3];
#pragma unroll
                for (int mi = 0; mi < MTW; ++mi)
#pragma unroll
                    for (int q = 0; q < 3; ++q) a[mi][q] = aw[u][mi][q];
                __builtin_amdgcn_sched_barrier(0);
                fetch(u);
                if (decltype(whole)::value || s0 + u < hi) products(u & 1, [&](int mi, int q) { return a[mi][q]; });
                convert((u + 1) % PF, (u + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int s0 = lo;
        for (; s0 + PF <= hi; s0 += PF) group(s0, std::true_type{});
        if (s0 < hi) group(s0, std::false_type{});
    }
    if constexpr (KSPLIT) {                                                 // each wave finishes the rows of four registers
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[0][r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[0][r] = ((red[0][4 * wave + r][lane] + red[1][4 * wave + r][lane]) + red[2][4 * wave + r][lane]) + red[3][4 * wave + r][lane];
    }
    int lane_hi = kh;                                                       // (opaque: the rows' addresses are not to be computed ahead of the contraction)
    asm volatile("" : "+v"(lane_hi));
    [[maybe_unused]] uint16_t* st = tiles[OUT ? wave : 0];
    auto tile = [&](auto index) {                                           // (a compile-time index: as a loop, eight tiles of this are not unrolled and the sums go to scratch)
        constexpr int mi = decltype(index)::value;
        if ((mt0 + mi) * 32 >= p.M) return;
        const int m0 = (mt0 + mi) * 32 + 4 * lane_hi + (KSPLIT ? 8 * wave : 0);
        if constexpr (WIDE) want(mi, lane_hi);
        if (!OUT && n >= p.N) return;
        auto finish = [&](float y, float b0, float s0, float e0) {
            y += pbias ? b0 : 0.0f;
            if (gelu) y = 0.5f * y * (1.0f + erff(y * 0.70710678118654752f));
            else if (noise) y = e0 + nz * y;
            else if (eb) { if (pscale) y *= s0; y = e0 + y; }
            return y;
        };
        float* y = pY + (size_t)b * p.M * p.ldy + n;
        // Three planes do not hold an infinity or a value past the largest bfloat16 (the planes of a product of two such cancel to NaN): a lane that sees a sum
        // which is not finite takes its rows again as the f32 kernels do, channel by channel
        float zero = 0.0f;
#pragma unroll
        for (int r = 0; r < NR; ++r) zero = fmaf(acc[mi][r], 0.0f, zero);
        if (zero != 0.0f && n < p.N) {
            const int T = TAPS ? P.ntaps : 1;
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                const int m = m0 + (r & 3) + 8 * (r >> 2);
                if (m >= p.M) break;
                float v = 0.0f;
#pragma unroll 1
                for (int i = 0; i < Kx * T; ++i) {                          // 16 channels, within them the taps, within a tap the channels
                    const int c = i / (16 * T) * 16 + (i & 15), j = i / 16 % T, t = TAPS ? n - p.pad + j * p.dil : n;
                    if (TAPS && (t < p.x_lo || t >= p.Tin)) continue;
                    float x = pX[((size_t)b * Kx + c) * p.ldx + t];
                    if constexpr (SNAKE) x = mis_snake(x, x6_ab[c], x6_ab[Kx + c]);
                    v = fmaf(pAT[((size_t)j * Kx + c) * p.M + m], x, v);
                    if (v != v) break;                                      // (NaN it stays)
                }
#pragma unroll
                for (int q = 0; q < NR; ++q) acc[mi][q] = q == r ? v : acc[mi][q];
            }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int m = m0 + (r & 3) + 8 * (r >> 2);
            acc[mi][r] = finish(acc[mi][r], bm[r], pscale ? sc[r] : 0.0f, eb ? e[r] : 0.0f);
            if ((!OUT || (pY && n < p.N)) && m < p.M) y[(size_t)m * p.ldy] = acc[mi][r];
        }
        if constexpr (OUT) {                                                // also (pY null: only) as the operand of the contraction behind
#pragma unroll
            for (int r0 = 0; r0 < 16; r0 += 8) {
                float o[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int m = m0 + 2 * r0 + (r & 3) + 8 * (r >> 2);
                    o[r] = acc[mi][r0 + r];
                    if (poa) o[r] = mis_snake(o[r], poa[m], pora[m]);
                }
                codec_tile_put<2>(o, st, r0, lane);
            }
            codec_tile_flush<2>(st, pout + (size_t)b * P.out.Tp * P.out.Cp + (mt0 + mi) * 32, P.out.stride, P.out.Cp, lane, [&](int c) {
                const int nn = n - (lane & 31) + c, r = nn - P.out.t_org;
                return nn < p.N && r < P.out.Tp ? r : -1;
            });
        }
    };
    x6_each(tile, std::make_integer_sequence<int, MTW>{});
    if constexpr (OUT) {                                                    // (the narrow form's other waves may be gone)
        if (wave == 0) codec_plane_ends(P.out, b, p.Tout, mt0 * 32, min(MTW * 32, p.M - mt0 * 32), bx == 0, bx == P.nbx - 1, lane, 64);
    }
}
template <int MTW, bool SNAKE, bool TAPS, bool WIDE, bool QUARTERS, bool OUT>
__global__ void __launch_bounds__(256, 2) k_x6_gemm(X6Gemm P, const uint16_t* wp) {
    x6_gemm_body<MTW, SNAKE, TAPS, WIDE, QUARTERS, OUT>(P, P.g.X, P.g.R, P.g.Y, P.g.bias, P.g.scale, P.g.noise, P.g.alpha, P.g.ralpha, P.g.AT, wp, P.out.alpha, P.out.ralpha, P.out.p);
}

template <bool SNAKE, bool TAPS, bool OUT>
static void launch_x6_gemm(X6Gemm P, const uint16_t* wp, int batch, hipStream_t s) {
    const GemmParams& p = P.g;
    P.nbx = (p.N + 127) / 128;
    const size_t sm = SNAKE ? (size_t)2 * p.K * sizeof(float) : 0;
    auto go = [&](auto kernel, int mtw) {
        P.my = (P.MT32 + mtw - 1) / mtw;
        P.tiles = P.nbx * P.my * batch;
        P.per = (P.tiles + 7) / 8;
        hipLaunchKernelGGL(kernel, dim3(8 * P.per), dim3(256), sm, s, P, wp);
    };
    // The form with the most rows per block (each converts its columns once) that still gives blocks enough; the same bits in all of them.  us:
    //   8 tiles / f32     256 x 256, 32 x 24576 columns 845 / 1133
    //   4 / 2 / 1         192 x 192, 18888 columns (296, 592 blocks of 4 and 2): 29 / 20 / 24; the same rows, two taps of 192 (K = 768): 105 / 72 / 102
    //   2 / 1 / f32       384 x 384 with Snake, 10160 columns: 41 / 56 / 71
    auto blocks = [&](int mtw) { return (int64_t)P.nbx * ((P.MT32 + mtw - 1) / mtw) * batch; };
    if constexpr (TAPS) {
        if (codec_quarters(p)) {
            // us, 4 tiles / 2 / the narrow form: 384 rows, K = 4608, 394 columns 204 / 155 / 31, 2368 columns (57, 114 blocks of 4 and 2) 204 / 154 / 91, eight such
            // rows (456, 912) 336 / 469 / 583; 128 rows, K = 3072, 16000 columns (250 of 2) 146 / 110 / 123; 192 rows, K = 1152, 18944 columns (296, 444) 94 / 71 / 97,
            // eight such rows 444 / 437 / 733; 768 rows, K = 9216, 296 columns 394 / 299 / 59 (f32: 94)
            // (strided convolutions of three taps then; on two, narrow: 384 rows, K = 3072, 2368 columns 72, 768 rows, K = 6144, 296 columns 45)
            if (P.MT32 > 2 && blocks(4) >= 384) go(k_x6_gemm<4, SNAKE, TAPS, true, true, false>, 4);
            else if (blocks(2) >= 192) go(k_x6_gemm<2, SNAKE, TAPS, true, true, false>, 2);
            else {
                P.nbx = (p.N + 31) / 32;
                go(k_x6_gemm<1, SNAKE, TAPS, false, true, false>, 1);
            }
            return;
        }
    }
    if (P.MT32 > 4 && blocks(8) >= 512) go(k_x6_gemm<8, SNAKE, TAPS, true, false, OUT>, 8);
    else if (P.MT32 > 2 && blocks(4) >= 512) go(k_x6_gemm<4, SNAKE, TAPS, true, false, OUT>, 4);
    else if (blocks(2) >= 256) go(k_x6_gemm<2, SNAKE, TAPS, true, false, OUT>, 2);
    else go(k_x6_gemm<1, SNAKE, TAPS, false, false, OUT>, 1);
}

bool launch_gemm_x6(int mode, bool snake, const GemmParams& p_in, int batch, hipStream_t s, const CodecPlanes* out) {
    GemmParams p = p_in;
    CodecPack* pack = p.pack ? p.pack : codec_x6_scope();
    const bool taps = mode == GEMM_TAPS;
    if (!pack || codec_exact_f32() || mode == GEMM_CONVT || (snake && (mode != GEMM_RESID || !p.alpha))) return false;
    const int Cin = taps ? p.Cin : p.K, ntaps = taps ? p.taps : 1;
    // By the matrix alone: a row's result must not depend on its length or its batch.  512 channels at one short row are bound by latency,
    // which the f32 kernel's four chunks of 64 channels in flight hide better (512 x 512, 96 columns: 15 us here, 8 there; 256 x 256, 768 columns: 11.3, 10.1);
    // a NoiseBlock of 64 channels is bound by memory (32 x 196608 columns: 918 us here, 842 there; 48 channels with residual, 37776 columns: 23, 34).
    if (p.M < (mode == GEMM_NOISE ? 96 : 48) || Cin < 32 || Cin % 16 || (!taps && Cin > 384)) return false;
    if (mode != GEMM_RESID && mode != GEMM_TAPS) p.R = p.scale = nullptr;
    MIS_REQUIRE(!out || codec_x6_writes_planes(mode, p, *out), MIS_ERR_GENERATION_FAILED, "codec contraction: %d rows for %d planes of %d channels", p.M, out->n, out->Cp);
    const CodecPack::X6& e = pack->get_x6(p.AT, ntaps, Cin, p.M, s);
    X6Gemm P{};
    P.g = p; P.mode = mode; P.ntaps = ntaps; P.nsteps = e.KS * ntaps; P.MT32 = e.MT32;
    if (out) P.out = *out;
    if (taps) launch_x6_gemm<false, true, false>(P, e.wp, batch, s);
    else if (out && snake) launch_x6_gemm<true, false, true>(P, e.wp, batch, s);
    else if (out) launch_x6_gemm<false, false, true>(P, e.wp, batch, s);
    else if (snake) launch_x6_gemm<true, false, false>(P, e.wp, batch, s);
    else launch_x6_gemm<false, false, false>(P, e.wp, batch, s);
    return true;
}

// ---- transposed convolution of stride 2, kernel 4 (two taps per phase), at most 64 rows ----------------------------------------------------
// Output 2 n + phase takes x[n + q] and x[n + q - 1], q = (phase + pad) / 2.  A block makes both phases of 126 columns n from 128 staged columns of x: Snake and
// the split run once per element (k_snac_convt: per phase and tap), the taps read the planes at column offsets, and a lane stores its two phases as one
// float2.  Chunks of 16 channels; weights of the four (phase, tap) pairs through LDS.  128 -> 64 channels, 32 x 98304 columns: 3.34 -> 1.44 ms (3.2 GB
// are 0.65 ms, the products 1.05); one row of 12288: 43 -> 27 us.
struct X6Noise { const float* noise; int rng; uint64_t key; const int32_t* row_ids; int64_t row_offset; };      // as in GemmParams
// NOISE: the NoiseBlock behind it, y = x + noise (W x), on the registers: a wave holds all rows of its columns, lanes l and l + 32 trade halves of x's planes, which
// makes them fragments, and W takes the place of the last chunk's weights (fragments [Cin / 16][MT][plane], the size of a chunk's).  As a launch of its own, in f32, it read and
// wrote the tensor: 16 us for one row of 24576 columns, 0.90 ms for 32 of 196608; here 3 us and 0.19 ms.
// x += nz (W x), x a phase's rows of a wave's columns.  SERIAL: a step's fragments at a time (where all of them do not fit the registers)
template <int MT, bool SERIAL>
__device__ __forceinline__ void x6_noise_block(f32x16_t (&acc)[MT], float nz, const x6_u4* As, int lane) {
    f32x16_t w[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int r = 0; r < 16; ++r) w[mi][r] = 0.0f;
    constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int ks = 0; ks < 2 * MT; ++ks) {
        float x[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) x[r] = acc[ks / 2][ks % 2 * 8 + r];
        bf16x8_t bv[3], av[MT][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) bv[q] = __builtin_bit_cast(bf16x8_t, codec_tile_piece(x, q == 0));
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int q = 0; q < 3; ++q) av[mi][q] = __builtin_bit_cast(bf16x8_t, As[((ks * MT + mi) * 3 + q) * 64 + lane]);
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int mi = 0; mi < MT; ++mi) w[mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi][QA[q]], bv[QB[q]], w[mi], 0, 0, 0);
        if constexpr (SERIAL) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mi][r] += nz * w[mi][r];
}
#define X6_CT 126
template <int MT, bool NOISE>
__device__ __forceinline__ void x6_convt_body(const GemmParams& p, const X6Noise& nb, const float* __restrict__ pX, float* __restrict__ pY, const float* __restrict__ pbias,
                                              const float* __restrict__ pa, const float* __restrict__ pra, const uint16_t* __restrict__ pwp, const uint16_t* __restrict__ pnw) {
    constexpr int APC = 4 * MT * 192, NA = APC / 256;
    __shared__ x6_u4 As[APC];
    __shared__ uint4 ts[3][2][128];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * X6_CT, b = blockIdx.y;
    const int q0 = p.pad / 2, dq = (1 + p.pad) / 2 - q0;                    // phase 1 reads dq columns further
    const int kg = wave >> 1, col = (wave & 1) * 64 + lane, t = n0 + q0 - 1 + col;
    const bool ok = t >= p.x_lo && t < p.Tin;
    const float* xb = pX + (size_t)b * p.Cin * p.ldx + min(max(t, p.x_lo), p.Tin - 1);
    f32x16_t acc[2][MT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const x6_u4* wsrc = reinterpret_cast<const x6_u4*>(pwp) + tid;
    float v[8];
    x6_u4 wv[NA];
    auto fetch = [&](int c0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = xb[(size_t)(c0 + kg * 8 + j) * p.ldx];
#pragma unroll
        for (int i = 0; i < NA; ++i) wv[i] = wsrc[(size_t)(c0 / 16) * APC + i * 256];
    };
    fetch(0);
    for (int c0 = 0; c0 < p.Cin; c0 += 16) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = c0 + kg * 8 + j;
            x[j] = ok ? mis_snake(v[j], pa[c], pra[c]) : 0.0f;               // (the padding is zero behind Snake as well)
        }
        uint4 h, m, l;
        x6_split<true>(x, h, m, l);
        __syncthreads();                                                    // the previous chunk's products are done
        ts[0][kg][col] = h; ts[1][kg][col] = m; ts[2][kg][col] = l;
#pragma unroll
        for (int i = 0; i < NA; ++i) As[tid + i * 256] = wv[i];
        if (c0 + 16 < p.Cin) fetch(c0 + 16);
        __syncthreads();
        constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int ph = 0; ph < 2; ++ph)
#pragma unroll
            for (int tap = 0; tap < 2; ++tap) {
                bf16x8_t bv[3];
                const int i = min(wave * 32 + (lane & 31) + 1 - tap + (ph ? dq : 0), 127);      // (past the end only for columns that are not stored)
#pragma unroll
                for (int q = 0; q < 3; ++q) bv[q] = *reinterpret_cast<const bf16x8_t*>(&ts[q][lane >> 5][i]);
                bf16x8_t av[MT][3];
#pragma unroll
                for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                    for (int q = 0; q < 3; ++q) av[mi][q] = __builtin_bit_cast(bf16x8_t, As[(((ph * 2 + tap) * MT + mi) * 3 + q) * 64 + lane]);
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi) acc[ph][mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi][QA[q]], bv[QB[q]], acc[ph][mi], 0, 0, 0);
            }
    }
    const int nl = wave * 32 + (lane & 31), n = n0 + nl, o = 2 * n;
    const bool in = nl < X6_CT && n < p.N && o < p.Tout;
    if (!NOISE && !in) return;
    const bool two = o + 1 < p.Tout, wide = two && !(p.ldy & 1) && !((uintptr_t)pY & 7), dup = n == 0 && p.dup_bias_n0;
    const float* bp = pbias ? pbias : pX;                                   // (loaded either way: a guard per value would be a round trip per value)
    const int btop = pbias ? p.M - 1 : 0;
    float nz[2] = {0.0f, 0.0f};
    if constexpr (NOISE) {
        x6_u4 nw[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i) nw[i] = reinterpret_cast<const x6_u4*>(pnw)[min(tid + i * 256, MT * MT * 2 * 192 - 1)];
        if (in && nb.noise) { nz[0] = nb.noise[(size_t)b * p.Tout + o]; nz[1] = two ? nb.noise[(size_t)b * p.Tout + o + 1] : 0.0f; }
        else if (in && nb.rng) {
            const uint64_t row = (uint64_t)(nb.row_offset + (nb.row_ids ? nb.row_ids[b] : b));
            nz[0] = codec_noise_value(nb.key, row, o); nz[1] = codec_noise_value(nb.key, row, o + 1);
        }
        __syncthreads();                                                    // the last chunk's products are done
#pragma unroll
        for (int i = 0; i < NA; ++i) As[tid + i * 256] = nw[i];
        __syncthreads();
    }
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int m0 = mi * 32 + 4 * (lane >> 5);
        float bm[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) bm[r] = bp[min(m0 + (r & 3) + 8 * (r >> 2), btop)];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float bv = pbias ? bm[r] : 0.0f;
#pragma unroll
            for (int ph = 0; ph < 2; ++ph) {
                acc[ph][mi][r] += bv;
                if (dup) acc[ph][mi][r] += bv;                              // streaming overlap-add counts the bias twice (GemmParams)
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NOISE) {
#pragma unroll
        for (int ph = 0; ph < 2; ++ph) x6_noise_block<MT, true>(acc[ph], nz[ph], As, lane);
        if (!in) return;
    }
    int hi = lane >> 5;                                                     // (opaque: the rows' addresses are not to be computed ahead)
    asm volatile("" : "+v"(hi));
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = mi * 32 + 4 * hi + (r & 3) + 8 * (r >> 2);
            float* y = pY + ((size_t)b * p.M + m) * p.ldy + o;
            if (m >= p.M) continue;
            if (wide) *reinterpret_cast<float2*>(y) = make_float2(acc[0][mi][r], acc[1][mi][r]);
            else { y[0] = acc[0][mi][r]; if (two) y[1] = acc[1][mi][r]; }
        }
}
template <int MT, bool NOISE>
__global__ void __launch_bounds__(256, 3) k_x6_convt(GemmParams p, X6Noise nb, const uint16_t* wp, const uint16_t* nw) {
    x6_convt_body<MT, NOISE>(p, nb, p.X, p.Y, p.bias, p.alpha, p.ralpha, wp, nw);
}

// The same for few blocks (the same bits): 62 columns a block, a wave makes one phase of 32 of them, chunks of 32 channels, two of them requested ahead.  With a block a compute unit at most, the chain
// of chunks is what there is to wait for: half as many, and none of them for its samples.  128 -> 64 channels
// with the NoiseBlock, one row of 12288 columns: 29.3 -> 20.9 us; a decode of 1 x 12 groups 352 -> 344, of 1 x 4 326 -> 317.
#define X6_CH 62
template <int MT, bool NOISE>
__device__ __forceinline__ void x6_convt_half_body(const GemmParams& p, const X6Noise& nb, const float* __restrict__ pX, float* __restrict__ pY, const float* __restrict__ pbias,
                                                   const float* __restrict__ pa, const float* __restrict__ pra, const uint16_t* __restrict__ pwp, const uint16_t* __restrict__ pnw) {
    constexpr int APC = 4 * MT * 192, NA = 2 * APC / 256, NN = MT * MT * 2 * 192;
    __shared__ x6_u4 As[2 * APC];
    __shared__ uint4 ts[3][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * X6_CH, b = blockIdx.y, ph = wave >> 1, cb = (wave & 1) * 32;
    const int q0 = p.pad / 2, dq = (1 + p.pad) / 2 - q0, t = n0 + q0 - 1 + lane;
    const bool ok = t >= p.x_lo && t < p.Tin;
    const float* xb = pX + ((size_t)b * p.Cin + wave * 8) * p.ldx + min(max(t, p.x_lo), p.Tin - 1);
    f32x16_t acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    const x6_u4* wsrc = reinterpret_cast<const x6_u4*>(pwp) + tid;
    const int chunks = p.Cin / 32;
    float v[2][8];
    x6_u4 wv[2][NA];
    auto fetch = [&](int slot, int c) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[slot][j] = xb[(size_t)(c * 32 + j) * p.ldx];
#pragma unroll
        for (int i = 0; i < NA; ++i) wv[slot][i] = wsrc[(size_t)c * 2 * APC + i * 256];
    };
    fetch(0, 0);
    fetch(1, min(1, chunks - 1));
    auto chunk = [&](int slot, int c) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int ch = c * 32 + wave * 8 + j;
            x[j] = ok ? mis_snake(v[slot][j], pa[ch], pra[ch]) : 0.0f;
        }
        uint4 h, m, l;
        x6_split<true>(x, h, m, l);
        __syncthreads();                                                    // the previous chunk's products are done
        ts[0][wave][lane] = h; ts[1][wave][lane] = m; ts[2][wave][lane] = l;
#pragma unroll
        for (int i = 0; i < NA; ++i) As[tid + i * 256] = wv[slot][i];
        if (c + 2 < chunks) fetch(slot, c + 2);
        __syncthreads();
        constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int tap = 0; tap < 2; ++tap) {
                bf16x8_t bv[3], av[MT][3];
                const int i = min(cb + (lane & 31) + 1 - tap + (ph ? dq : 0), 63);             // (past the end only for columns that are not stored)
#pragma unroll
                for (int q = 0; q < 3; ++q) bv[q] = *reinterpret_cast<const bf16x8_t*>(&ts[q][2 * k + (lane >> 5)][i]);
#pragma unroll
                for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                    for (int q = 0; q < 3; ++q) av[mi][q] = __builtin_bit_cast(bf16x8_t, As[k * APC + (((ph * 2 + tap) * MT + mi) * 3 + q) * 64 + lane]);
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi) acc[mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi][QA[q]], bv[QB[q]], acc[mi], 0, 0, 0);
            }
    };
    for (int c = 0; c < chunks; c += 2) {
        chunk(0, c);
        if (c + 1 < chunks) chunk(1, c + 1);
    }
    const int nl = cb + (lane & 31), n = n0 + nl, o = 2 * n + ph;
    const bool in = nl < X6_CH && n < p.N && o < p.Tout, dup = n == 0 && p.dup_bias_n0;
    const float* bp = pbias ? pbias : pX;
    const int btop = pbias ? p.M - 1 : 0;
    float nz = 0.0f;
    if constexpr (NOISE) {
        if (in && nb.noise) nz = nb.noise[(size_t)b * p.Tout + o];
        else if (in && nb.rng) nz = codec_noise_value(nb.key, (uint64_t)(nb.row_offset + (nb.row_ids ? nb.row_ids[b] : b)), o);
        __syncthreads();                                                    // the last chunk's products are done
        for (int i = tid; i < NN; i += 256) As[i] = reinterpret_cast<const x6_u4*>(pnw)[i];
        __syncthreads();
    }
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int m0 = mi * 32 + 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float bm = bp[min(m0 + (r & 3) + 8 * (r >> 2), btop)], bv = pbias ? bm : 0.0f;
            acc[mi][r] += bv;
            if (dup) acc[mi][r] += bv;
        }
    }
    if constexpr (NOISE) x6_noise_block<MT, false>(acc, nz, As, lane);
    if (!in) return;
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = mi * 32 + 4 * (lane >> 5) + (r & 3) + 8 * (r >> 2);
            if (m < p.M) pY[((size_t)b * p.M + m) * p.ldy + o] = acc[mi][r];
        }
}
template <int MT, bool NOISE>
__global__ void __launch_bounds__(256, 1) k_x6_convt_half(GemmParams p, X6Noise nb, const uint16_t* wp, const uint16_t* nw) {
    x6_convt_half_body<MT, NOISE>(p, nb, p.X, p.Y, p.bias, p.alpha, p.ralpha, wp, nw);
}

bool launch_convt_x6(const GemmParams& p, int batch, hipStream_t s, const GemmParams* noise) {
    CodecPack* pack = p.pack ? p.pack : codec_x6_scope();
    if (!pack || codec_exact_f32() || p.s != 2 || p.K != 2 * p.Cin || p.M > 64 || p.M < 32 || p.Cin % 16 || !p.alpha) return false;
    // (a NoiseBlock of as many rows as the tiles have and of this row's whole output)
    if (noise && (noise->M != p.M || noise->K != p.M || p.M % 32 || noise->N != p.Tout || noise->bias)) return false;
    const uint16_t* wp = pack->get_x6(p.AT, 4, p.Cin, p.M, s).wp;           // [phase][tap][Cin][M]
    const uint16_t* nw = noise ? pack->get_x6(noise->AT, 1, p.M, p.M, s).wp : nullptr;
    const X6Noise nb = noise ? X6Noise{noise->noise, noise->noise_rng, noise->noise_key, noise->row_ids, noise->row_offset} : X6Noise{};
#define X6_GO(K, W) do { \
        const dim3 grid((p.N + W - 1) / W, batch); \
        if (p.M > 32 && noise) hipLaunchKernelGGL((K<2, true>), grid, dim3(256), 0, s, p, nb, wp, nw); \
        else if (p.M > 32) hipLaunchKernelGGL((K<2, false>), grid, dim3(256), 0, s, p, nb, wp, nw); \
        else if (noise) hipLaunchKernelGGL((K<1, true>), grid, dim3(256), 0, s, p, nb, wp, nw); \
        else hipLaunchKernelGGL((K<1, false>), grid, dim3(256), 0, s, p, nb, wp, nw); } while (0)
    // (while each has a compute unit of its own: a decode of 2 x 12 groups, 396 blocks, 427 either way)
    if (p.Cin % 32 == 0 && (int64_t)((p.N + X6_CH - 1) / X6_CH) * batch <= 256) X6_GO(k_x6_convt_half, X6_CH);
    else X6_GO(k_x6_convt, X6_CT);
#undef X6_GO
    return true;
}
