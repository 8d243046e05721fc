// codec_bf3.hip - split-bf16 dense contractions for the codec decoders (SNAC / DAC / Qwen3-TTS speech tokenizer / Vocos / EnCodec).
//
// The codec weights and activations are f32 (SNAC ships f32 checkpoints; the waveform gate is 1e-4 RMS), and gfx950 has no TF32-like
// MFMA: exact-f32 MFMA runs at 1/16 of the bf16 rate.  Here every f32 operand is split into two bf16 halves, x = xh + xl with
// xh = bf16(x), xl = bf16(x - xh) (relative error of the pair <= 2^-18), and a product becomes three bf16 MFMAs accumulated in f32:
// xh.wh + xh.wl + xl.wh (the lo.lo term, <= 2^-16 of the product, is dropped).  Measured on the CPU emulation of exactly this
// arithmetic inside the SNAC oracle (tools/bf16x3_emulation.py, profiles/r02_bf16x3_emulation.json): 1.06e-5 RMS on the 24 kHz decode
// against the 1e-4 gate (plain bf16: 5.7e-3).  The f32-accurate kernels (codec_x6.hip, codec_f32.hip, snac.hip) stay: encoders (codebook
// decisions), small or memory-bound shapes, and MIS_CODEC_EXACT_F32=1.
//
// Three kernels:
//   k_bf3_pack_w   A^T f32 [taps][Cin][M] -> MFMA-A fragments of v_mfma_f32_32x32x16_bf16, hi and lo, [tap][M/32][Cp/16][hl][64][8]
//                  (once per weight matrix, cached per model in CodecPack)
//   k_bf3_split    activation pre-pass: (Snake) -> split -> transpose to time-major planes xh, xl [B][Tp][Cp] with zero pads, so that a
//                  B fragment (8 consecutive channels of one time column) is one aligned 16-byte piece; Snake runs ONCE per element
//                  (the staged f32 kernels re-run it per 64-row block and per transposed-conv phase)
//   k_bf3_gemm     128 x 128 output tile per block (64 x 128 or 64 x 64 where that gives few blocks): 4 MFMA waves (64 x 64 each) + 1 loader wave.  The loader streams the activation
//                  tile (with its tap halo) by LDS-DMA into an NBUF-deep ring, chunk = 32 channels, running NBUF-1 chunks ahead on its
//                  OWN vmcnt counter; the MFMA waves take the packed weight fragments straight from L2 into registers (prefetched two
//                  to seven steps ahead) and the activation fragments from LDS (XOR-swizzled at the DMA source, conflict-free ds_read_b128).
//                  One s_barrier per chunk.  Taps (dense k-tap convs), transposed-conv phases and 1x1 convs share the tile code:
//                  tap j reads the staged tile at a column offset.
//
// Between two contractions the planes come from the epilogue in front (launch_gemm_chain): Snake and the split run there, on registers, and the pre-pass - a launch, a read and a
// write of the tensor - is gone, with the f32 tensor where nothing else reads it.  DAC, one row of 30 / 250 frames, four of 400: 951 / 1688 / 8060 -> 748 / 1472 / 7490 us.
// An operand may have three planes instead (NP = 3, the arithmetic and the bits of codec_x6.hip): the strided convolutions of SNAC's encoder, whose phase split writes them
// (k_enc_phase_planes; k_x6_gemm converts a column once per block of rows: 96 / 192 / 384 / 768 rows of one recording of 151111 samples 46 + 52 + 71 + 44 us, 33 + 39 + 46 + 31 here, and
// 7 more in the phase splits), and the 1x1 contractions of 193 .. 384 channels behind Snake, which k_x6_gemm converts
// once per 64 rows (384 x 384, 10005 columns: 45 us, 52 with planes out; 34 here).  Of up to 192 channels k_pw_x6 converts once in all and reads four bytes, not six: 192 channels,
// 40021 columns: 42 us there, 43 here and 4 more in front; 96, 80043 columns: 36 and 41.
#include "common.h"
#include "codec_kernels.h"

#define B3_BM 128
#define B3_KC 32
#define B3_THREADS 320

typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

struct Bf3Params {
    GemmParams g;
    const uint16_t* wp;
    const uint16_t* xp;   // planes [plane][B][Tp][Cp]
    size_t xplane;        // elements of one plane
    size_t wtap, wmt, wks;                // weight fragments: elements from a tap, a row tile, a 16-channel step to the next
    CodecPlanes out;      // .p: the output (also) as the planes of the contraction behind it
    int mode, ntaps, MT32, Cp, Tp, t_org;
    int ksplit;           // > 1: a tile has that many blocks; a block contracts chunks [nchunks slice / ksplit, nchunks (slice + 1) / ksplit)
    float* part;          //      and writes its raw float32 sums to part[slice][b][M][ldy] (k_bf3_splitk_epilogue finishes)
    int batch;
    int nbx, my, inner, per, tiles;       // column tiles, row tiles, phases or K slices of a tile, tiles per XCD, all tiles
};


// ---- weights: A^T [ntaps][Cin][M] f32 -> fragments --------------------------------------------------------------------------------
__global__ void k_bf3_pack_w(const float* __restrict__ AT, uint16_t* __restrict__ wp, int ntaps, int Cin, int M, int MT32, int KS) {
    const size_t total = (size_t)ntaps * MT32 * KS * 512;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const int j = (int)(e & 7), lane = (int)((e >> 3) & 63);
        size_t r = e >> 9;
        const int ks = (int)(r % KS); r /= KS;
        const int mt = (int)(r % MT32);
        const int tap = (int)(r / MT32);
        const int m = mt * 32 + (lane & 31), c = ks * 16 + (lane >> 5) * 8 + j;
        float v = (m < M && c < Cin) ? AT[((size_t)tap * Cin + c) * M + m] : 0.0f;
        const uint16_t h = f32_to_bf16(v);
        const uint16_t l = f32_to_bf16(v - bf16_to_f32(h));
        const size_t o = ((((size_t)tap * MT32 + mt) * KS + ks) * 2) * 512 + (size_t)lane * 8 + j;
        wp[o] = h;
        wp[o + 512] = l;
    }
}

// ---- activations: x f32 [B][C][ldx] -> planes [B][Tp][Cp] (column t' holds input column t' + t_org; zero outside [x_lo, Tin)) ---------
// Block: 64 columns x SP_CB channels.  A wave reads 64 consecutive columns of eight channels at a time (all its 32 loads are requested before the first use:
// one memory round trip), splits them and writes one 16-byte piece per plane to LDS; stores are coalesced along channels (16-byte pieces, a full
// SP_CB-channel row per 16 threads).  Channel by channel under its guard it was 32 round trips of latency: 663 -> 297 us for 32 x 98304 columns of 256 channels
// (1.6 GB: 5.4 TB/s), 17.9 -> 9.2 us for 2080 columns of 768
#define SP_CB 128
#define SP_LD (SP_CB + 8)             // LDS row stride in bf16 (272 B: 16-byte aligned rows, 4 banks apart: eight lanes' 16-byte writes cover 32 banks)
__global__ void __launch_bounds__(256) k_bf3_split(const float* __restrict__ X, uint16_t* __restrict__ xh, uint16_t* __restrict__ xl,
                                                   const float* __restrict__ alpha, const float* __restrict__ ralpha,
                                                   int C, int ldx, int x_lo, int Tin, int Cp, int Tp, int t_org) {
    __shared__ __attribute__((aligned(16))) uint16_t sh[64 * SP_LD], sl[64 * SP_LD];
    const int tl = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);       // (scalar: the channels' parameters come by s_load)
    const int tp0 = blockIdx.x * 64, c0 = blockIdx.y * SP_CB, b = blockIdx.z;
    const int cw = min(SP_CB, Cp - c0);                         // channels of this block (multiple of 32)
    const int t = tp0 + tl + t_org;
    const bool tin = tp0 + tl < Tp && t >= x_lo && t < Tin;
    const float* xb = X + (int64_t)b * C * ldx + (tin ? t : 0);
    constexpr int NO = SP_CB / 32;                              // octets of channels per wave
    float v[NO][8];
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[o][j] = xb[(int64_t)min(c0 + (wave + 4 * o) * 8 + j, C - 1) * ldx];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const int cc = (wave + 4 * o) * 8;
        if (cc >= cw) continue;
        uint32_t h[4], l[4];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            float x[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int c = c0 + cc + j + i;
                x[i] = v[o][j + i];
                if (alpha) x[i] = mis_snake(x[i], alpha[min(c, C - 1)], ralpha[min(c, C - 1)]);
                x[i] = tin && c < C ? x[i] : 0.0f;
            }
            h[j / 2] = (uint32_t)f32_to_bf16(x[0]) | ((uint32_t)f32_to_bf16(x[1]) << 16);
            l[j / 2] = (uint32_t)f32_to_bf16(x[0] - __uint_as_float(h[j / 2] << 16)) | ((uint32_t)f32_to_bf16(x[1] - __uint_as_float(h[j / 2] & 0xffff0000u)) << 16);
        }
        *reinterpret_cast<uint4*>(sh + tl * SP_LD + cc) = make_uint4(h[0], h[1], h[2], h[3]);
        *reinterpret_cast<uint4*>(sl + tl * SP_LD + cc) = make_uint4(l[0], l[1], l[2], l[3]);
    }
    __syncthreads();
    const int pieces = cw / 8;                                  // 16-byte pieces per row
    for (int i = threadIdx.x; i < 64 * pieces; i += 256) {
        const int r = i / pieces, pc = i - r * pieces;
        if (tp0 + r >= Tp) continue;
        const size_t o = ((size_t)b * Tp + tp0 + r) * Cp + c0 + pc * 8;
        *reinterpret_cast<uint4*>(xh + o) = *reinterpret_cast<const uint4*>(sh + r * SP_LD + pc * 8);
        *reinterpret_cast<uint4*>(xl + o) = *reinterpret_cast<const uint4*>(sl + r * SP_LD + pc * 8);
    }
}

// ---- the contraction -----------------------------------------------------------------------------------------------------------------
template <int NP, int MI> struct Bf3A { bf16x8_t v[MI][NP]; };     // [m tile][plane]
template <int NP, int NI> struct Bf3B { bf16x8_t v[NI][NP]; };     // [n tile][plane]

// One step's order: an MFMA with a weight load behind it, then one with a tile read, then the rest (sched_group_barrier masks: 0x008 MFMA, 0x002 VALU,
// 0x020 VMEM read, 0x100 DS read)
template <int NV, int ND, int NM> __device__ __forceinline__ void bf3_interleave() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    }
}

// One output of a three-plane contraction as the f32 kernels make it: 16 channels, within them the taps (a column each), within a tap the channels; NaN it stays
__device__ __forceinline__ float bf3_retake(const uint16_t* __restrict__ x, size_t plane, int Cp, const float* __restrict__ at, int Cin, int M, int ntaps) {
    float v = 0.0f;
#pragma unroll 1
    for (int i = 0; i < Cin * ntaps && v == v; ++i) {
        const int c = i / (16 * ntaps) * 16 + (i & 15), j = i / 16 % ntaps;
        const uint16_t* q = x + (size_t)j * Cp + c;
        const float hm = bf16_to_f32(q[0]) + bf16_to_f32(q[plane]);
        v = fmaf(at[((size_t)j * Cin + c) * M], fabsf(hm) < INFINITY ? hm + bf16_to_f32(q[2 * plane]) : hm, v);
    }
    return v;
}

// The body takes the arrays the epilogue touches as restrict-qualified PARAMETERS: GemmParams is a struct, clang ignores restrict on
// struct members, and without it every bias / residual load of the epilogue waits behind the previous row's store (the same effect
// cost the fused unit kernel of snac.hip 25 %).
template <int NP, int MI, int NI, int NQ, int NBUF, int NTAPS, int AR, bool QUARTERS, bool OUT>
__device__ __forceinline__ void bf3_body(const Bf3Params& P, const float* __restrict__ pX, const float* __restrict__ pR, float* __restrict__ pY,
                                         const float* __restrict__ pbias, const float* __restrict__ pscale, const float* __restrict__ pnoise,
                                         const float* __restrict__ poa, const float* __restrict__ pora, uint16_t* __restrict__ pout) {
    constexpr int PLANE = NQ * 512;                       // bf16 per plane: NQ DMA instructions of 1 KiB (16 columns x 32 channels)
    constexpr int BUF = NP * PLANE;
    constexpr int NST = 2 * NTAPS;                        // MFMA steps (16 channels of one tap) per chunk
    constexpr int CG = NST % AR == 0 ? 1 : (2 * NST) % AR == 0 ? 2 : (3 * NST) % AR == 0 ? 3 : 4;      // chunks per straight-line group: whole turns of the weight ring
    static_assert(CG * NST % AR == 0 && CG * NST % 2 == 0, "registers rotate in whole turns");
    constexpr int BN = 64 * NI, NPROD = NP == 2 ? 3 : 6, ND = NPROD * MI * NI - NP * MI < NP * NI ? NPROD * MI * NI - NP * MI : NP * NI;
    static_assert(!OUT || NBUF * BUF >= 4 * NI * CP_LDS(3), "the ring holds the waves' output tiles");
    static_assert((NBUF - 2) * NP * NQ < 64, "the loader's wait counts the younger chunks");
    __shared__ __attribute__((aligned(1024))) uint16_t lds[NBUF * BUF];
    const GemmParams& p = P.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // blocks are dealt to the XCDs by id mod 8: an XCD takes a contiguous range of tiles, all row tiles of a column tile in a row and all phases of a tile in
    // a row, so that its L2 holds their activation tile and merges the phases' interleaved stores (M = 128, K = 2 x 256, 4 phases, 32 x 24576 columns: 2.03 ->
    // 1.68 ms; where the phases' weights, 34 MB for M = 512, K = 2 x 1024, 8 phases, are more than it holds: 0.57 -> 0.60, 0.80 with the phases outside)
    const int xi = blockIdx.x >> 3, in = xi % P.inner, tileid = (blockIdx.x & 7) * P.per + xi / P.inner;
    if (tileid >= P.tiles) return;
    const int by = tileid % P.my, bxb = tileid / P.my, bx = bxb % P.nbx, b = bxb / P.nbx;
    int phase = 0, sh0 = 0, dsh = 0, tapbase = 0, slice = 0;
    if (P.mode == GEMM_CONVT) { phase = in; sh0 = (phase + p.pad) / p.s; dsh = -1; tapbase = phase * NTAPS; }
    else if (P.mode == GEMM_TAPS) { sh0 = -p.pad; dsh = p.dil; }
    if (P.ksplit > 1) slice = in;
    const int shmin = min(sh0, sh0 + (NTAPS - 1) * dsh);
    const int nchunks_all = P.Cp / B3_KC;
    const int c_lo = P.ksplit > 1 ? nchunks_all * slice / P.ksplit : 0;                        // this block's chunks (split-K: a slice of them)
    const int nchunks = (P.ksplit > 1 ? nchunks_all * (slice + 1) / P.ksplit : nchunks_all) - c_lo;
    const int n0 = bx * BN;

    if (wave == 4) {
        // ---- loader: tile column i = input column n0 + shmin + i.  DMA instruction q moves columns 16q .. 16q+15, four lanes per column;
        // lane slot gs holds channel group gs ^ ((i >> 2) & 3) (the swizzle is on the SOURCE address, the LDS side of a DMA is lane-linear)
        const int il = lane >> 2, grp = (lane & 3) ^ ((il >> 2) & 3);
        const size_t col0 = ((size_t)b * P.Tp + (size_t)(n0 + shmin - P.t_org + il)) * P.Cp + grp * 8;
        const uint16_t* sx = P.xp + col0 + (size_t)c_lo * B3_KC;
        const size_t qstride = (size_t)16 * P.Cp;
        auto issue = [&](int cc) {
            const uint16_t* h = sx + cc * B3_KC;
            const int buf = cc % NBUF;
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int i = 0; i < NP; ++i)
                    __builtin_amdgcn_global_load_lds((gptr_t)(h + q * qstride + i * P.xplane), (lptr_t)&lds[buf * BUF + i * PLANE + q * 512], 16, 0, 0);
        };
        for (int c = 0; c < NBUF - 1 && c < nchunks; ++c) issue(c);
        for (int cc = 0; cc < nchunks; ++cc) {
            // chunk cc must have landed; up to NBUF-2 younger chunks stay in flight
            if (nchunks - 1 - cc >= NBUF - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * NP * NQ) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            if (cc + NBUF - 1 < nchunks) issue(cc + NBUF - 1);
        }
        return;
    }

    // ---- MFMA waves: 2 x 2, wave tile MI x NI tiles of 32 x 32
    const int wm = wave >> 1, wn = wave & 1;
    const int mt0 = (by * 2 + wm) * MI;
    if (mt0 >= P.MT32) {                                   // no rows for this wave (M <= 64 in this block row): keep the barrier count
        for (int cc = 0; cc < nchunks; ++cc) __builtin_amdgcn_s_barrier();
        return;
    }
    f32x16_t acc[MI][NI];

    // weight stream: step (chunk, tap, ks) -> fragments of the row tiles, hi and lo.  It runs AR - 1 steps ahead of the MFMAs, across
    // chunk boundaries (it does not depend on the staged tile).  A second row tile past M re-reads the first (its rows are
    // never stored).  The body below is CG chunks (CG * NST steps) of straight-line code: the weight registers rotate with period AR,
    // the tile-fragment registers with period 2, every index is a compile-time constant and there is no branch between the MFMAs,
    // so the waitcnt pass keeps exactly the AR - 2 younger weight loads in flight (with branches in the body it fell back to vmcnt(0)).
    const uint16_t* wbase = P.wp + (size_t)lane * 8 + (size_t)tapbase * P.wtap + (size_t)mt0 * P.wmt + (size_t)c_lo * 2 * P.wks;
    const size_t mt1 = (mt0 + 1 < P.MT32) ? P.wmt : 0;
    const int ncol = wn * 32 * NI + (lane & 31), kgrp = lane >> 5;
    Bf3A<NP, MI> aq[AR];
    Bf3B<NP, NI> bq[2];
    auto loadA = [&](Bf3A<NP, MI>& f, int chunk, int tap, int ks) {
        chunk = min(chunk, nchunks - 1);                     // the last steps prefetch past the end: re-read the last chunk
        const uint16_t* q = wbase + (size_t)tap * P.wtap + (size_t)(chunk * 2 + ks) * P.wks;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int i = 0; i < NP; ++i) f.v[mi][i] = *reinterpret_cast<const bf16x8_t*>(q + (mi ? mt1 : 0) + i * 512);
    };
    auto readB = [&](Bf3B<NP, NI>& f, const uint16_t* tile, int tap, int ks) {
        const int toff = sh0 + tap * dsh - shmin;
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            const int i = ncol + ni * 32 + toff;
            const uint16_t* q = tile + i * 32 + (((ks * 2 + kgrp) ^ ((i >> 2) & 3)) * 8);
#pragma unroll
            for (int j = 0; j < NP; ++j) f.v[ni][j] = *reinterpret_cast<const bf16x8_t*>(q + j * PLANE);
        }
    };
    // products per tile pair, two planes: hi.hi, hi.lo, lo.hi; three: the six of codec_x6.hip, smallest first; MI * NI independent accumulators between dependent MFMAs
    auto products = [&](const Bf3A<NP, MI>& A, const Bf3B<NP, NI>& B) {
        constexpr int QA[2][6] = {{0, 0, 1}, {2, 0, 1, 1, 0, 0}}, QB[2][6] = {{0, 1, 0}, {0, 2, 1, 0, 1, 0}};
#pragma unroll
        for (int term = 0; term < (NP == 2 ? 3 : 6); ++term) {
            const int ta = QA[NP - 2][term], tb = QB[NP - 2][term];
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v[mi][ta], B.v[ni][tb], acc[mi][ni], 0, 0, 0);
        }
    };
    // a chunk's steps: tap by tap; three planes: 16 channels at a time, within them the taps (k_x6_gemm's order)
    constexpr auto TAP = [](int t) { return NP == 2 ? t >> 1 : t % NTAPS; };
    constexpr auto KSTEP = [](int t) { return NP == 2 ? t & 1 : t / NTAPS; };
#pragma unroll
    for (int J = 0; J < AR - 1; ++J) loadA(aq[J], J / NST, TAP(J % NST), KSTEP(J % NST));
    const uint16_t* tile = lds;
    int gbuf = 0;                                           // ring slot of the next chunk
    const float* Xb = pX + (size_t)b * p.Cin * p.ldx;
    const bool convt = P.mode == GEMM_CONVT, gelu = !OUT && P.mode == GEMM_GELU, noise = !OUT && P.mode == GEMM_NOISE;
    const float* Rr = (convt || gelu || noise) ? nullptr : pR;
    constexpr bool EARLY = OUT && MI == 1 && NTAPS == 1;
    float early[EARLY ? NI : 1][EARLY ? 16 : 1];
    if constexpr (EARLY) {
        if (Rr) {
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    early[ni][r] = Rr[((size_t)b * p.M + min(mt0 * 32 + (r & 3) + 8 * (r >> 2) + 4 * kgrp, p.M - 1)) * p.ldy + min(n0 + (wn * NI + ni) * 32 + (lane & 31), p.N - 1)];
        }
    }

    {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        int cc = 0;
        f32x16_t tot[QUARTERS ? MI : 1][QUARTERS ? NI : 1];
        [[maybe_unused]] auto close_quarter = [&](bool first) {              // (a sum that starts at 0 is never -0: the first may be taken over)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        tot[QUARTERS ? i : 0][QUARTERS ? j : 0][r] = first ? acc[i][j][r] : tot[QUARTERS ? i : 0][QUARTERS ? j : 0][r] + acc[i][j][r];
                        acc[i][j][r] = 0.0f;
                    }
        };
        [[maybe_unused]] int quarter = 1;
        static_assert(!QUARTERS || CG == 1, "a quarter ends where a group does");
        for (; cc + CG <= nchunks; cc += CG) {
            if constexpr (QUARTERS) {
                if (quarter < 4 && cc == nchunks * quarter / 4) { close_quarter(quarter == 1); ++quarter; }
            }
#pragma unroll
            for (int I = 0; I < CG * NST; ++I) {
                const int t = I % NST;
                if (t == 0) {
                    __builtin_amdgcn_s_barrier();
                    tile = lds + gbuf * BUF;
                    gbuf = gbuf + 1 == NBUF ? 0 : gbuf + 1;
                    readB(bq[I & 1], tile, 0, 0);
                }
                // one scheduling region per step: the prefetches of later steps cannot sink out of it (left alone the scheduler moves
                // them next to their use), and inside it they are spread over the shadows of the MFMAs instead of running ahead
                // of them with the matrix pipe idle: MFMA, then a weight load or a tile read with its address arithmetic
                __builtin_amdgcn_sched_barrier(0);
                if (t + 1 < NST) readB(bq[(I + 1) & 1], tile, TAP(t + 1), KSTEP(t + 1));
                const int J = I + AR - 1;
                loadA(aq[J % AR], cc + J / NST, TAP(J % NST), KSTEP(J % NST));
                products(aq[I % AR], bq[I & 1]);
                bf3_interleave<NP * MI, ND, NPROD * MI * NI - NP * MI - ND>();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // tail: up to CG - 1 chunks, same schedule with a runtime bound (rotation phase 0 here)
        if (CG > 1 && cc < nchunks) {
            const int rem = (nchunks - cc) * NST;
#pragma unroll
            for (int I = 0; I < (CG - 1) * NST; ++I) {
                if (I < rem) {
                    const int t = I % NST;
                    if (t == 0) {
                        __builtin_amdgcn_s_barrier();
                        tile = lds + gbuf * BUF;
                        gbuf = gbuf + 1 == NBUF ? 0 : gbuf + 1;
                        readB(bq[I & 1], tile, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + 1 < NST) readB(bq[(I + 1) & 1], tile, TAP(t + 1), KSTEP(t + 1));
                    const int J = I + AR - 1;
                    loadA(aq[J % AR], cc + J / NST, TAP(J % NST), KSTEP(J % NST));
                    products(aq[I % AR], bq[I & 1]);
                    bf3_interleave<NP * MI, ND, NPROD * MI * NI - NP * MI - ND>();
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }

        if constexpr (QUARTERS) {
            close_quarter(false);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = tot[i][j];
        }
        // ---- epilogue (the modes of k_codec_gemm / k_conv_taps / k_snac_convt).  C/D layout: col = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
        // opaque: left visible, the 32 rows' 64-bit offsets are computed ahead of the main loop and spilled (860 B of scratch per
        // lane in the multi-tile experiment: 1.9x slower)
        int lane_hi = lane >> 5;
        asm volatile("" : "+v"(lane_hi));
        if (P.ksplit > 1) {                                  // split-K: the raw sums of this slice; k_bf3_splitk_epilogue adds the slices up
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const int n = n0 + (wn * NI + ni) * 32 + (lane & 31);
                if (n >= p.N) continue;
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int m = (mt0 + mi) * 32 + (r & 3) + 8 * (r >> 2) + 4 * lane_hi;
                        if (m < p.M) P.part[(((size_t)slice * P.batch + b) * p.M + m) * p.ldy + n] = acc[mi][ni][r];
                    }
                }
            }
            return;
        }
        if constexpr (NP == 3) {
            // Three planes hold an infinity as one beside a NaN: a lane that sees a sum which is not finite takes its rows again as the f32 kernels do
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    const int n = n0 + (wn * NI + ni) * 32 + (lane & 31);
                    float zero = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) zero = fmaf(acc[mi][ni][r], 0.0f, zero);
                    if (zero == 0.0f || n >= p.N) continue;
#pragma unroll 1
                    for (int r = 0; r < 16; ++r) {
                        const int m = (mt0 + mi) * 32 + (r & 3) + 8 * (r >> 2) + 4 * lane_hi;
                        const float v = m < p.M ? bf3_retake(P.xp + ((size_t)b * P.Tp + (n + sh0 - P.t_org)) * P.Cp, P.xplane, P.Cp, p.AT + m, p.Cin, p.M, NTAPS) : 0.0f;
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[mi][ni][q] = q == r ? v : acc[mi][ni][q];
                    }
                }
        }
        if constexpr (OUT) {
            // the output as the operand of the contraction behind this one (its pre-pass's values), and in f32 where something else reads it; the ring is free by now.
            // Eight rows at a time, their values (the residual's of both column tiles too) requested together; EARLY: the residual came with the first weights
            __syncthreads();
            uint16_t* st = lds + wave * NI * CP_LDS(3);
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
                const int mt = (mt0 + mi) * 32;
                if (mt >= p.M) break;
#pragma unroll
                for (int r0 = 0; r0 < 16; r0 += 8) {
                    const int m0 = mt + 2 * r0 + 4 * lane_hi;
                    float bm[8], al[8], ra[8], e[NI][8];
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        const int m = m0 + (r & 3) + 8 * (r >> 2);
                        bm[r] = pbias ? pbias[m] : 0.0f;
                        if (poa) { al[r] = poa[m]; ra[r] = pora[m]; }
                        if (Rr && !EARLY) {
#pragma unroll
                            for (int ni = 0; ni < NI; ++ni) e[ni][r] = Rr[((size_t)b * p.M + m) * p.ldy + min(n0 + (wn * NI + ni) * 32 + (lane & 31), p.N - 1)];
                        }
                    }
#pragma unroll
                    for (int ni = 0; ni < NI; ++ni) {
                        const int n = n0 + (wn * NI + ni) * 32 + (lane & 31), o = convt ? p.s * n + phase : n;
                        float y[8];
#pragma unroll
                        for (int r = 0; r < 8; ++r) {
                            y[r] = acc[mi][ni][r0 + r] + bm[r];
                            if (convt && n == 0 && p.dup_bias_n0) y[r] += bm[r];
                            if (Rr) y[r] += EARLY ? early[EARLY ? ni : 0][EARLY ? r0 + r : 0] : e[ni][r];
                        }
                        if (pY && n < p.N && o < p.Tout) {
#pragma unroll
                            for (int r = 0; r < 8; ++r) pY[((size_t)b * p.M + m0 + (r & 3) + 8 * (r >> 2)) * p.ldy + o] = y[r];
                        }
                        if (poa) {
#pragma unroll
                            for (int r = 0; r < 8; ++r) y[r] = mis_snake(y[r], al[r], ra[r]);
                        }
                        if (P.out.n == 3) codec_tile_put<3>(y, st + ni * CP_LDS(3), r0, lane);
                        else codec_tile_put<2>(y, st + ni * CP_LDS(3), r0, lane);
                    }
                }
                uint16_t* d = pout + (size_t)b * P.out.Tp * P.out.Cp + mt;
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    auto row = [&](int c) {
                        const int n = n0 + (wn * NI + ni) * 32 + c, o = convt ? p.s * n + phase : n, r = o - P.out.t_org;
                        return n < p.N && o < p.Tout && r < P.out.Tp ? r : -1;
                    };
                    if (P.out.n == 3) codec_tile_flush<3>(st + ni * CP_LDS(3), d, P.out.stride, P.out.Cp, lane, row);
                    else codec_tile_flush<2>(st + ni * CP_LDS(3), d, P.out.stride, P.out.Cp, lane, row);
                }
            }
            if (phase == 0) codec_plane_ends(P.out, b, p.Tout, mt0 * 32, min(MI * 32, p.M - mt0 * 32), bx == 0 && wn == 0, bx == P.nbx - 1 && wn == 1, lane, 64);
            return;
        }
        // a tile's bias and residual (or NoiseBlock input) values are requested together, clamped; one by one under their guards each was a round trip
        const float* eb = noise ? Xb : Rr ? Rr + (size_t)b * p.M * p.ldy : nullptr;
        const int lde = noise ? p.ldx : p.ldy;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            const int m0 = (mt0 + mi) * 32 + 4 * lane_hi;
            float bm[16], sc[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) bm[r] = pbias ? pbias[min(m0 + (r & 3) + 8 * (r >> 2), p.M - 1)] : 0.0f;
            if (Rr && pscale) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = pscale[min(m0 + (r & 3) + 8 * (r >> 2), p.M - 1)];
            }
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const int n = n0 + (wn * NI + ni) * 32 + (lane & 31);
                float e[16];
                if (eb) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) e[r] = eb[(size_t)min(m0 + (r & 3) + 8 * (r >> 2), p.M - 1) * lde + min(n, p.N - 1)];
                }
                float nz = 0.0f;
                if (noise && n < p.N) {
                    if (pnoise) nz = pnoise[(size_t)b * p.N + n];
                    else if (p.noise_rng) nz = codec_noise_value(p.noise_key, (uint64_t)(p.row_offset + (p.row_ids ? p.row_ids[b] : b)), n);
                }
                const int o = convt ? p.s * n + phase : n;
                if (n >= p.N || o >= p.Tout) continue;
                const bool dupb = convt && n == 0 && p.dup_bias_n0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + (r & 3) + 8 * (r >> 2);
                    float v = acc[mi][ni][r] + bm[r];
                    if (dupb) v += bm[r];
                    if (gelu) v = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));
                    if (Rr) { if (pscale) v *= sc[r]; v += e[r]; }
                    if (noise) v = e[r] + nz * v;
                    if (m < p.M) pY[((size_t)b * p.M + m) * p.ldy + o] = v;
                }
            }
        }
    }
}

template <int NP, int MI, int NI, int NQ, int NBUF, int NTAPS, int AR, int MINW, bool QUARTERS, bool OUT>
__global__ void __launch_bounds__(B3_THREADS, MINW) k_bf3_gemm(Bf3Params P) {
    bf3_body<NP, MI, NI, NQ, NBUF, NTAPS, AR, QUARTERS, OUT>(P, P.g.X, P.g.R, P.g.Y, P.g.bias, P.g.scale, P.g.noise, P.out.alpha, P.out.ralpha, P.out.p);
}

// split-K: Y = epilogue(sum over slices in slice order + bias) - the 1x1 modes' epilogues of bf3_body (plain / GELU / residual with scale).  xp: three planes, whose sums
// that are not finite are taken again (taps at consecutive columns)
__global__ void k_bf3_splitk_epilogue(const float* __restrict__ part, int S, int batch, int mode, const float* __restrict__ bias, const float* __restrict__ scale,
                                      const float* __restrict__ R, float* __restrict__ Y, int M, int N, int ldy, const uint16_t* __restrict__ xp, size_t xplane, int Tp, int Cp,
                                      const float* __restrict__ at, int Cin, int ntaps) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x, m = blockIdx.y, b = blockIdx.z;
    if (n >= N) return;
    const size_t rowo = ((size_t)b * M + m) * ldy;
    float v = 0.0f;
    for (int s = 0; s < S; ++s) v += part[(((size_t)s * batch + b) * M + m) * ldy + n];
    if (xp && !(fabsf(v) < INFINITY)) v = bf3_retake(xp + ((size_t)b * Tp + n) * Cp, xplane, Cp, at + m, Cin, M, ntaps);
    v += bias ? bias[m] : 0.0f;
    if (mode == GEMM_GELU) v = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));
    if (mode == GEMM_RESID && R) { if (scale) v *= scale[m]; v += R[rowo + n]; }
    Y[rowo + n] = v;
}

// ---- host side ------------------------------------------------------------------------------------------------------------------------
CodecPack::~CodecPack() {
    for (auto& e : entries) if (e.wp) (void)hipFree(e.wp);
    for (auto& e : x6) if (e.wp) (void)hipFree(e.wp);
}

const CodecPack::Entry& CodecPack::get(const float* at, int ntaps, int Cin, int M, hipStream_t s) {
    for (auto& e : entries)
        if (e.at == at && e.ntaps == ntaps && e.Cin == Cin && e.M == M) return e;
    Entry e{};
    e.at = at; e.ntaps = ntaps; e.Cin = Cin; e.M = M;
    e.Cp = (Cin + B3_KC - 1) / B3_KC * B3_KC;
    e.KS = e.Cp / 16;
    e.MT32 = (M + 31) / 32;
    const size_t n = (size_t)ntaps * e.MT32 * e.KS * 1024;
    HIP_CHECK(hipMalloc((void**)&e.wp, n * sizeof(uint16_t)));
    hipLaunchKernelGGL(k_bf3_pack_w, dim3((unsigned)std::min<size_t>((n / 2 + 255) / 256, 8192)), dim3(256), 0, s, at, e.wp, ntaps, Cin, M, e.MT32, e.KS);
    entries.push_back(e);
    return entries.back();
}

static thread_local CodecPack *tl_pack = nullptr, *tl_x6 = nullptr;
CodecPackScope::CodecPackScope(CodecPack* p, bool bf3) : prev(tl_pack), prev_x6(tl_x6) { tl_pack = bf3 ? p : nullptr; tl_x6 = p; }
CodecPackScope::~CodecPackScope() { tl_pack = prev; tl_x6 = prev_x6; }

static int bf3_env(const char* name, int dflt) {
    const char* v = getenv(name);
    return v ? atoi(v) : dflt;
}

CodecPack* codec_x6_scope() { return tl_x6; }
bool codec_exact_f32() { return bf3_env("MIS_CODEC_EXACT_F32", 0) != 0; }

// What the two-plane contractions take.  What pays: MFMA-bound shapes.  A 1x1 conv over few channels is HBM-bound and the pre-pass would only add traffic
// (measured per dispatch, profiles/r02_codec/: 1x1 over <= 512 channels and the last SNAC transposed conv, M*K = 16 K,
// are faster on the exact-f32 kernels; every 7-tap conv and the transposed convs from M*K = 36 K up gain 2.3 - 4x)
struct Bf3Shape { int ntaps, Cin, span, t_org, wtaps, phases, extra, parts; bool three; };      // three: planes (the caller's)
static bool bf3_shape(int mode, const GemmParams& p, Bf3Shape& h) {
    const bool one = mode == GEMM_PLAIN || mode == GEMM_GELU || mode == GEMM_RESID || mode == GEMM_NOISE;
    h = Bf3Shape{1, p.K, 0, 0, 1, 1, 0, 1, false};
    if (mode == GEMM_TAPS && p.taps == 2 && codec_quarters(p)) h.parts = 4;
    if (mode == GEMM_TAPS) { h.ntaps = p.taps; h.Cin = p.Cin; h.span = (p.taps - 1) * p.dil; h.t_org = -p.pad; h.wtaps = p.taps; }
    else if (mode == GEMM_CONVT) {
        if (p.Cin <= 0 || p.K % p.Cin || p.K / p.Cin > 2) return false;
        h.ntaps = p.K / p.Cin;                                       // 2: kernel 2s (overlap-add); 1: kernel = stride (A^T holds one tap)
        h.Cin = p.Cin; h.span = h.ntaps - 1; h.wtaps = h.ntaps * p.s; h.phases = p.s;
        h.t_org = p.pad / p.s - (h.ntaps - 1);                       // phase 0 has the smallest q = (phase + pad) / s
        h.extra = (p.s - 1 + p.pad) / p.s - p.pad / p.s;             // the phases share one operand: columns from the smallest shift of any phase to the largest
        if (h.extra > 1) return false;
    } else if (!one) return false;
    return p.M >= 32 && h.span <= 64 && (h.ntaps == 1 || h.ntaps == 2 || h.ntaps == 7);
}
static bool bf3_takes(int mode, const GemmParams& p, const Bf3Shape& h) {
    const int min_k1 = bf3_env("MIS_BF3_MIN_K1", 768), min_k = bf3_env("MIS_BF3_MIN_K", 32), min_mk = bf3_env("MIS_BF3_MIN_MK_CONVT", 32768);
    if (mode == GEMM_CONVT) return h.Cin >= min_k && (int64_t)p.M * p.K >= min_mk;
    return h.Cin >= (mode == GEMM_TAPS ? min_k : min_k1);
}
bool bf3_takes_convt(const GemmParams& p) {
    Bf3Shape h;
    return (p.pack || tl_pack) && !codec_exact_f32() && bf3_shape(GEMM_CONVT, p, h) && bf3_takes(GEMM_CONVT, p, h);
}
// Tile: 128 x 128 (64 x 64 per wave); 64 x 128 while those are at most 128 blocks - half of the chip idle, each block one serial chain of chunks -
// and 64 x 64 while 64 x 128 still are (or no more than 64 columns exist).  The same bits: the order of the products of an output does not change.
// The small tiles run alone on a compute unit, with registers to spare: weights seven (not two) steps ahead, which covers a trip to HBM.
// us, 128 x 128 / 64 x 128 / 64 x 64: 768 rows, 7 taps of 768, 2080 columns: 102 / 60 / 79; 768 rows, K = 768: 51 / 24 / 26;
// 1536 rows, 7 taps of 1024, 250 columns: 140 / 70 / 55; SNAC, one row of 12 groups: 48 / - / 19, 41 / 22 / 15, 33 / - / 14, 29 / 17 / 16.
// A quarter of K a block (three planes, two taps of at least 512 channels): counted as the blocks they are, 64 x 64 up to 256 of 64 x 128 (us, 64 x 128 / 64 x 64: 384 rows,
// K = 3072, 2361 columns, 456 blocks: 40 / 45; 768 rows, K = 6144, 296 columns, 144: 36 / 26; k_x6_gemm: 71, 44), and always for rows of at most 64 columns (that one,
// rows of 4 columns, 8: 67 / 41, 64: 371 / 268; of 24, 8: 68 / 42; k_x6_gemm: 43, 439, 43).
struct Bf3Tile { bool few; int NI, nbx, nq, Tp; };
static Bf3Tile bf3_tile(const GemmParams& p, const Bf3Shape& h, int batch) {
    const int nb128 = (p.N + 127) / 128;
    Bf3Tile t{};
    t.few = (int64_t)nb128 * ((p.M + B3_BM - 1) / B3_BM) * batch * h.phases * h.parts <= 128;
    t.NI = (h.three && h.parts > 1 && p.N <= 64) || (t.few && (p.N <= 64 || (int64_t)nb128 * ((p.M + 63) / 64) * batch * h.phases * h.parts <= (h.parts > 1 ? 256 : 128))) ? 1 : 2;
    t.nbx = (p.N + 64 * t.NI - 1) / (64 * t.NI);
    t.nq = 4 * t.NI + (h.span == 0 ? 0 : h.span <= 16 ? 1 : 4);
    t.Tp = (t.nbx - 1) * 64 * t.NI + t.nq * 16 + h.extra;
    return t;
}
// Three planes, where the epilogue in front writes them: 1x1 contractions with Snake and a residual that k_x6_gemm would convert for itself
static bool bf3_three(int mode, const GemmParams& p) { return mode == GEMM_RESID && p.alpha && p.M >= 48 && p.K > 192 && p.K <= 384; }

// memory for planes; where there is none left the caller goes on without them
static bool planes_fit(CodecPack& pack, int slot, size_t n, size_t spare) {
    if (pack.plain) return false;
    DevBuf<uint16_t>& b = pack.planes[slot];
    if (b.p && n <= b.n) return true;
    for (const size_t more : {spare, (size_t)0}) {
        try { b.alloc(n + more); return true; }
        catch (const MisNoMemory&) { if (!more) return false; }
    }
    return false;
}

// Strided convolutions of the encoders, on two taps of the phase split: three planes, written by k_enc_phase_planes
bool codec_planes_strided(const GemmParams& p, int batch, CodecPlanes& out) {
    CodecPack* pack = codec_x6_scope();
    Bf3Shape h;
    if (!pack || codec_exact_f32() || p.taps != 2 || p.dil != 1 || p.pad != 0 || p.Cin % 32 || p.M < 48 || !bf3_shape(GEMM_TAPS, p, h)) return false;
    h.three = true;
    const Bf3Tile t = bf3_tile(p, h, batch);
    out = CodecPlanes{};
    out.n = 3; out.Cp = h.Cin; out.Tp = t.Tp;
    out.stride = (size_t)batch * t.Tp * h.Cin;
    if (!planes_fit(*pack, 0, 3 * out.stride, 3 * out.stride / 8)) return false;                  // (the convolutions behind take as much, but for their tiles' ends)
    out.p = pack->planes[0].p;
    return true;
}

// (the planes a contraction takes; the memory is codec_planes')
static bool codec_planes_shape(int mode, bool snake, const GemmParams& p, int batch, CodecPlanes& out) {
    Bf3Shape h;
    if (!(p.pack ? p.pack : tl_pack) || codec_exact_f32() || !bf3_shape(mode, p, h) || h.Cin % 32) return false;
    const bool two = bf3_takes(mode, p, h);
    if (!two && !(snake && bf3_three(mode, p))) return false;
    const Bf3Tile t = bf3_tile(p, h, batch);
    out = CodecPlanes{};
    out.n = two ? 2 : 3; out.Cp = h.Cin; out.Tp = t.Tp; out.t_org = h.t_org; out.ends = h.span > 0 || h.extra > 0;
    out.stride = (size_t)batch * t.Tp * h.Cin;
    if (snake) { out.alpha = p.alpha; out.ralpha = p.ralpha; }
    return true;
}
bool codec_planes(int mode, bool snake, const GemmParams& p, int batch, int slot, CodecPlanes& out) {
    if (!codec_planes_shape(mode, snake, p, batch, out)) return false;
    CodecPack* pack = p.pack ? p.pack : tl_pack;
    if (!planes_fit(*pack, slot, out.n * out.stride, 0)) return false;
    out.p = pack->planes[slot].p;
    return true;
}

bool bf3_writes_planes(int mode, const GemmParams& p) { return p.M % 32 == 0 && !p.split_k_ok && !p.scale && (mode == GEMM_TAPS || mode == GEMM_CONVT || mode == GEMM_PLAIN || mode == GEMM_RESID); }

bool launch_gemm_bf3(int mode, bool snake, const GemmParams& p_in, int batch, hipStream_t s, const CodecPlanes* in, const CodecPlanes* out) {
    GemmParams p = p_in;
    if (!p.pack) p.pack = tl_pack;
    if (!p.pack || codec_exact_f32()) return false;
    Bf3Shape h;
    if (!bf3_shape(mode, p, h) || (!in && !bf3_takes(mode, p, h))) return false;
    if (out) {
        MIS_REQUIRE(bf3_writes_planes(mode, p) && out->Cp == p.M && !(in && in->n == 3 && h.ntaps == 2), MIS_ERR_GENERATION_FAILED, "codec contraction: %d rows for an operand of %d channels", p.M, out->Cp);
    }
    const int ntaps = h.ntaps, Cin = h.Cin, span = h.span;
    const bool three = h.three = in && in->n == 3;
    const Bf3Tile t = bf3_tile(p, h, batch);
    const bool few = t.few;
    const int NI = t.NI, nb128 = (p.N + 127) / 128;
    Bf3Params P{};
    P.g = p; P.g.Cin = Cin;
    P.mode = mode; P.ntaps = ntaps; P.Tp = t.Tp; P.t_org = h.t_org;
    if (three) {
        const CodecPack::X6& e = p.pack->get_x6(p.AT, h.wtaps, Cin, p.M, s);
        P.wp = e.wp; P.MT32 = e.MT32;
        P.wmt = 1536; P.wtap = (size_t)e.MT32 * 1536; P.wks = h.wtaps * P.wtap;
    } else {
        const CodecPack::Entry& e = p.pack->get(p.AT, h.wtaps, Cin, p.M, s);
        P.wp = e.wp; P.MT32 = e.MT32;
        P.wks = 1024; P.wmt = (size_t)e.KS * 1024; P.wtap = e.MT32 * P.wmt;
    }
    P.Cp = (Cin + B3_KC - 1) / B3_KC * B3_KC;
    if (in) { P.xp = in->p; P.xplane = in->stride; }
    else {
        P.xplane = (size_t)batch * t.Tp * P.Cp;
        DevBuf<uint16_t>& xs = p.pack->planes[out && out->p == p.pack->planes[0].p ? 1 : 0];
        xs.alloc(2 * P.xplane);
        P.xp = xs.p;
        const bool sn = snake && p.alpha;
        hipLaunchKernelGGL(k_bf3_split, dim3((t.Tp + 63) / 64, (P.Cp + SP_CB - 1) / SP_CB, batch), dim3(256), 0, s, p.X, xs.p, xs.p + P.xplane,
                           sn ? p.alpha : nullptr, sn ? p.ralpha : nullptr, Cin, p.ldx, p.x_lo, p.Tin, P.Cp, t.Tp, h.t_org);
    }
    if (out) P.out = *out;
    // launch-shaped 1x1 contractions (Soprano's ConvNeXt GEMMs at 257 frames: 18 or 54 blocks per row of a 256-CU part, 60 us per launch):
    // the K range split over blocks.  The factor is a function of the SHAPE of one batch row only (a row's bits do not depend on the batch
    // it shares); float32 slabs, summed in slice order by k_bf3_splitk_epilogue
    const int nchunks = P.Cp / B3_KC, per_row = nb128 * ((p.M + B3_BM - 1) / B3_BM);
    int ksplit = 1;
    if (p.split_k_ok && ntaps == 1 && (mode == GEMM_PLAIN || mode == GEMM_GELU || mode == GEMM_RESID) && !bf3_env("MIS_BF3_NO_SPLITK", 0)) {
        if (per_row <= 32 && nchunks >= 32) ksplit = 4;
        else if (per_row <= 64 && nchunks >= 16) ksplit = 2;
    }
    // Three planes, K >= 1024: four partial sums in every form (codec_quarters), in blocks of their own while that is what fills the chip (tiles of 64 columns: always)
    const bool quarters = three && ntaps == 2 && codec_quarters(p);
    if (quarters && (NI == 1 || (int64_t)t.nbx * ((p.M + 63) / 64) * batch < 512)) ksplit = 4;
    if (ksplit > 1) {
        p.pack->part.alloc((size_t)ksplit * batch * p.M * p.ldy);
        P.ksplit = ksplit; P.part = p.pack->part.p; P.batch = batch;
    }
    // Rows that are no multiple of 128 leave a wave row of the large tile without any, and its blocks (7 taps: one a compute unit) come in whole rounds: 64 x 128 there,
    // two blocks a compute unit.  us, 128 x 128 / 64 x 128: 192 rows, 7 taps, 40000 columns 91 / 63, 2 taps (5 phases) 62 / 54; 96 rows, 80000 columns 67 / 45, 47 / 39;
    // whole tiles: 384 rows, 7 taps, 10000 columns 60 / 64, 2 taps of 512 .. 128 rows (SNAC, 32 rows) 588 / 767, 1395 / 1748, 1734 / 1966
    const bool half = !few && (three || (ntaps != 1 && p.M % B3_BM != 0));
    const int bm = few || half ? 64 : B3_BM;
    P.nbx = t.nbx; P.my = (p.M + bm - 1) / bm; P.inner = h.phases * ksplit;
    P.tiles = P.nbx * P.my * batch; P.per = (P.tiles + 7) / 8;
    const dim3 grid(8 * P.per * P.inner), block(B3_THREADS);
#define B3_RUN(...) hipLaunchKernelGGL((k_bf3_gemm<__VA_ARGS__>), grid, block, 0, s, P)
#define B3_GO(...) do { if (out) B3_RUN(__VA_ARGS__, false, true); else B3_RUN(__VA_ARGS__, false, false); } while (0)
    if (three && ntaps == 2) {
        if (NI == 1) B3_RUN(3, 1, 1, 5, 5, 2, 6, 2, false, false);
        else if (quarters && ksplit == 1) B3_RUN(3, 1, 2, 9, 4, 2, 4, 2, true, false);
        else B3_RUN(3, 1, 2, 9, 2, 2, 4, 3, false, false);
    }
    else if (three) {
        if (NI == 1) B3_GO(3, 1, 1, 4, 6, 1, 6, 2);
        else B3_GO(3, 1, 2, 8, 3, 1, 4, 3);
    }
    else if (few && NI == 1) {
        if (ntaps == 1) B3_GO(2, 1, 1, 4, 8, 1, 8, 2);
        else if (ntaps == 2) B3_GO(2, 1, 1, 5, 8, 2, 8, 2);
        else if (span <= 16) B3_GO(2, 1, 1, 5, 4, 7, 7, 2);
        else B3_GO(2, 1, 1, 8, 4, 7, 7, 2);
    } else if (few) {
        if (ntaps == 1) B3_GO(2, 1, 2, 8, 5, 1, 8, 2);
        else if (ntaps == 2) B3_GO(2, 1, 2, 9, 5, 2, 8, 2);
        else if (span <= 16) B3_GO(2, 1, 2, 9, 4, 7, 7, 2);
        else B3_GO(2, 1, 2, 12, 4, 7, 7, 2);
    }
    else if (half && ntaps == 2) B3_GO(2, 1, 2, 9, 4, 2, 4, 3);
    else if (half && span <= 16) B3_GO(2, 1, 2, 9, 4, 7, 4, 3);
    else if (half) B3_GO(2, 1, 2, 12, 3, 7, 4, 3);
    // MINW 3 = two blocks (ten waves) per CU, 168 registers: fits 1 and 2 taps; the 7-tap body would spill (measured 2.3x slower), so it
    // runs one block per CU (a persistent loop over column tiles was measured too: no gain, profiles/r02_codec/ab_record.json)
    else if (ntaps == 1) B3_GO(2, 2, 2, 8, 4, 1, 3, 3);
    else if (ntaps == 2) B3_GO(2, 2, 2, 9, 4, 2, 3, 3);
    else if (span <= 16) B3_GO(2, 2, 2, 9, 4, 7, 4, 2);
    else B3_GO(2, 2, 2, 12, 4, 7, 4, 2);
#undef B3_GO
#undef B3_RUN
    if (ksplit > 1)
        hipLaunchKernelGGL(k_bf3_splitk_epilogue, dim3((p.N + 255) / 256, p.M, batch), dim3(256), 0, s, P.part, ksplit, batch, mode, p.bias, p.scale, p.R, p.Y, p.M,
                           p.N, p.ldy, three ? P.xp : nullptr, P.xplane, P.Tp, P.Cp, p.AT, Cin, ntaps);
    return true;
}

void launch_gemm_chain(const CodecOp* ops, int n, int batch, hipStream_t s) {
    CodecPlanes cur{}, nxt{};
    bool have = false;
    // (the largest of each turn first: a buffer that grows along the chain waits for the device at every step of its first pass)
    int top[2] = {-1, -1};
    size_t most[2] = {0, 0};
    for (int i = 0; i + 1 < n; ++i)
        if (codec_planes_shape(ops[i + 1].mode, ops[i + 1].snake, ops[i + 1].g, batch, nxt) && nxt.n * nxt.stride > most[i & 1]) { most[i & 1] = nxt.n * nxt.stride; top[i & 1] = i + 1; }
    for (int slot = 0; slot < 2; ++slot)
        if (top[slot] >= 0) codec_planes(ops[top[slot]].mode, ops[top[slot]].snake, ops[top[slot]].g, batch, slot, nxt);
    for (int i = 0; i < n; ++i) {
        const CodecOp& o = ops[i];
        const bool want = i + 1 < n && codec_planes(ops[i + 1].mode, ops[i + 1].snake, ops[i + 1].g, batch, i & 1, nxt);
        if (have) {
            GemmParams g = o.g;
            if (!g.ldx) g.ldx = g.Tin;
            if (!g.ldy) g.ldy = g.Tout;
            if (!g.R) g.scale = nullptr;
            const bool outs = want && bf3_writes_planes(o.mode, g);
            if (outs && !o.keep) g.Y = nullptr;
            MIS_REQUIRE(launch_gemm_bf3(o.mode, o.snake, g, batch, s, &cur, outs ? &nxt : nullptr), MIS_ERR_GENERATION_FAILED, "codec contraction refused its own operand");
            have = outs;
        } else
            have = launch_gemm(o.mode, o.snake, o.g, batch, s, want ? &nxt : nullptr, o.keep);
        cur = nxt;
    }
}

extern "C" mis_status mis_debug_codec_chain(int device, int n, int channels, int batch, int columns, const float* x, const float* wt, const float* bias, const float* alpha, const float* ralpha,
                                            float* y_out) {
    MIS_API_BEGIN
    MIS_REQUIRE(n >= 1 && channels >= 32 && channels % 32 == 0 && batch >= 1 && columns >= 1 && x && wt && bias && alpha && ralpha && y_out, MIS_ERR_INVALID_INPUT, "bad argument");
    HIP_CHECK(hipSetDevice(device));
    const size_t C = channels, elems = C * batch * columns;
    CodecPack pack;
    DevBuf<float> w, v[3], buf[2];                                   // matrices; biases, Snake's parameters; tensors in turns
    w.alloc(n * C * C); v[0].alloc(n * C); v[1].alloc(C); v[2].alloc(C);
    for (auto& b : buf) b.alloc(elems);
    HIP_CHECK(copy_now(w.p, wt, n * C * C * 4, hipMemcpyHostToDevice));
    HIP_CHECK(copy_now(v[0].p, bias, n * C * 4, hipMemcpyHostToDevice));
    std::vector<float> ap(channels);
    for (int i = 0; i < channels; ++i) ap[i] = snake_alpha(alpha[i]);
    HIP_CHECK(copy_now(v[1].p, ap.data(), C * 4, hipMemcpyHostToDevice));
    HIP_CHECK(copy_now(v[2].p, ralpha, C * 4, hipMemcpyHostToDevice));
    HIP_CHECK(copy_now(buf[0].p, x, elems * 4, hipMemcpyHostToDevice));
    std::vector<CodecOp> ops;
    for (int i = 0; i < n; ++i) {
        GemmParams g{};
        g.AT = w.p + i * C * C; g.bias = v[0].p + i * C; g.alpha = v[1].p; g.ralpha = v[2].p;
        g.X = g.R = buf[i & 1].p; g.Y = buf[(i + 1) & 1].p;
        g.M = g.K = channels; g.N = g.Tin = g.Tout = columns;
        ops.push_back({GEMM_RESID, true, true, g});
    }
    {
        CodecPackScope scope(&pack);
        launch_gemm_chain(ops.data(), n, batch, hipStreamPerThread);
    }
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(copy_now(y_out, buf[n & 1].p, elems * 4, hipMemcpyDeviceToHost));
    MIS_API_END
}
