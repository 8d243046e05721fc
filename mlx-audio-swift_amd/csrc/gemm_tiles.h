// gemm_tiles.h - bf16 matrix products on tiles of 32 TM x 256 outputs, four waves, one persistent block a compute unit.
//
// What bounds a bf16 product on this part once its operands come from L2 is the LDS: a compute unit reads 128 bytes a cycle, and the eight waves of a
// 256 x 256 tile with 64 x 128 outputs each ask for 192 KB of fragments a k-step of 64 (1536 cycles, and 512 for the LDS-DMA that fills the
// buffers) beside 2048 cycles of MFMA.  Four waves with 128 x 16 TM outputs each read 128 KB; a wave then has a SIMD's 512 registers for itself
// (accumulators in the AGPRs, two halves of a k-step's fragments in VGPRs), and nothing but its own instruction order overlaps its work:
//   * the fragments of the next half are requested between the MFMAs of this one, every S-th instruction, and have arrived when it ends;
//   * a k-step has ONE barrier, in its middle: behind it the buffer just read is refilled (NBUF - 1 k-steps ahead) and the next one is read;
//   * MFMAs, LDS reads and waits are asm statements, so that their order is the one written here and the accumulators stay where they are
//     (with the builtins hipcc moved 200 of them between the register files every k-step: 855 against 1103 TFLOP/s);
//   * the block goes on to its next tile without a gap: the last k-steps of a tile request the first ones of the next, the epilogue runs meanwhile.
// Measured (8192^3, us): TM 8 862, TM 6 903, TM 5 903, TM 4 924 - 1275 .. 1190 TFLOP/s; torch.matmul 935.  Smaller TM are there because tiles come in whole
// rounds of 256 blocks (the callers choose).  Products are added in the order of k: the bits of k_gemm_pf and k_gemm_big2 / 3.
#pragma once
#include "common.h"

// The tiles are numbered in bands of G row tiles, row tiles fastest, and an XCD (blocks are dealt to the XCDs by id mod 8) takes one range of them: the 32
// blocks it runs together share G row tiles of X and 32 / G column tiles of W in its L2.
struct TileOrder {
    int mt, nt;
    __device__ __forceinline__ void at(int G, int t, int& mi, int& ni) const {
        const int band = t / (G * nt), left = t - band * G * nt, rows = min(G, mt - band * G);
        ni = left / rows;
        mi = band * G + left - ni * rows;
    }
};

__device__ __forceinline__ uint32_t gt_lds_offset(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }

// Wave (wn, wm) = (wave >> 1, wave & 1) holds W rows 128 wn + 16 i and X rows 16 TM wm + 16 j of the tile in acc[i][j] (the MFMA's C/D layout).
// PACKED: W as the decode step's tiles [N/16][K/32][64][8], a fragment 1 KB lane-linear in memory and in LDS; else rows of K elements, their 16-byte
// pieces swizzled on the way to LDS.  X: rows.  K: a multiple of 64, NBUF k-steps at least.  Offsets are 32-bit: operands of less than 2^31 elements.
template <int TM, bool PACKED>
struct GemmTiles {
    static constexpr int TN = 8, BN = 256, BM = 32 * TM, BK = 64, QW = 8, QX = TM, NQ = QW + QX;
    static constexpr int WB = BN * BK * 2, XB = BM * BK * 2, STEP = WB + XB;       // bytes of a k-step
    static constexpr int NBUF = STEP * 3 <= 160 * 1024 ? 3 : 2;
    static constexpr int LDS = NBUF * STEP;

    // tiles first, first + stride, ... < tiles.  woff(t, q, lane): element offset of the lane's 16 bytes of the tile's q-th KB of W at k = 0; xoff(t, r): of row r
    // of its X; epi(t, acc) stores a finished tile
    // operands(t, W, X): the two operands of tile t
    template <class FO, class FW, class FX, class FE>
    static __device__ __forceinline__ void run(unsigned char* lds, int K, int first, int stride, int tiles, FO operands, FW woff, FX xoff, FE epi) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave >> 1, wm = wave & 1;
        const int KS = K / BK;
        uint32_t off[NQ];                                            // bytes
        const bf16_t *Wb, *Xb;
        auto point = [&](int t) {
            operands(t, Wb, Xb);
            int ln = lane;
            asm volatile("" : "+v"(ln));                             // (computed here for each tile: hoisted, these take the registers that TM = 8 has not got)
#pragma unroll
            for (int q = 0; q < QW; ++q) off[q] = 2 * (uint32_t)woff(t, wave * QW + q, ln);
#pragma unroll
            for (int q = 0; q < QX; ++q) {
                const int r = (wave * QX + q) * 8 + (ln >> 3);
                off[QW + q] = 2 * ((uint32_t)xoff(t, r) + ((ln & 7) ^ ((r >> 1) & 7)) * 8);
            }
        };
        auto stage1 = [&](int buf, int ks, int n) {                  // the n-th LDS load of a k-step
            unsigned char* l = lds + buf * STEP;
            const unsigned char* src = n < QW ? reinterpret_cast<const unsigned char*>(Wb) + (size_t)ks * (PACKED ? 2048 : 128) : reinterpret_cast<const unsigned char*>(Xb) + (size_t)ks * 128;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off[n]),
                                             (__attribute__((address_space(3))) void*)(l + (n < QW ? (wave * QW + n) * 1024 : WB + (wave * QX + n - QW) * 1024)), 16, 0, 0);
        };
        const int sw = (lane >> 1) & 7;
        const uint32_t base = gt_lds_offset(lds);
        const uint32_t p0 = ((lane >> 4) ^ sw) * 16, p1 = ((4 + (lane >> 4)) ^ sw) * 16;
        // fragment i of half h: PACKED image [16 n-tiles][2][1 KB] lane-linear, else rows of 128 bytes, swizzled
        const uint32_t w0 = base + (PACKED ? wn * TN * 2048 + lane * 16 : (wn * TN * 16 + (lane & 15)) * 128 + p0);
        const uint32_t w1 = base + (PACKED ? wn * TN * 2048 + 1024 + lane * 16 : (wn * TN * 16 + (lane & 15)) * 128 + p1);
        const uint32_t x0 = base + WB + (wm * TM * 16 + (lane & 15)) * 128 + p0;
        const uint32_t x1 = base + WB + (wm * TM * 16 + (lane & 15)) * 128 + p1;
        bf16x8_t a[2][TN], b[2][TM];
        auto read = [&](int n, uint32_t w, uint32_t x, bf16x8_t (&fa)[TN], bf16x8_t (&fb)[TM]) {        // the n-th fragment of a half: X first
            if (n < TM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[n < TM ? n : 0]) : "v"(x), "n"((n < TM ? n : 0) * 2048) : "memory");
            else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[n < TM ? 0 : n - TM]) : "v"(w), "n"((n < TM ? 0 : n - TM) * 2048) : "memory");
        };
        auto bind = [&](bf16x8_t (&fa)[TN], bf16x8_t (&fb)[TM]) {
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0]) :: "memory");
#pragma unroll
            for (int i = 1; i < TN; ++i) asm volatile("" : "+v"(fa[i]));
#pragma unroll
            for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(fb[j]));
        };
        constexpr int NF = TN + TM, S = TM > 6 ? 3 : 2;             // fragments of a half; one is requested behind every S-th MFMA
        static_assert(NF == NQ && NF * S <= TN * TM, "every request of a half stands between its MFMAs");
        f32x4_t acc[TN][TM];
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        int t = first, buf = 0;
        point(t);
#pragma unroll
        for (int i = 0; i < NBUF; ++i)
#pragma unroll
            for (int n = 0; n < NQ; ++n) stage1(i, i, n);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 1) * NQ) : "memory");
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int n = 0; n < NF; ++n) read(n, w0, x0, a[0], b[0]);
        auto step = [&](int kn) {                                    // multiplies the k-step in `buf`, requests step kn behind it
            const int nb = buf + 1 == NBUF ? 0 : buf + 1;
            const uint32_t wo = w1 + buf * STEP, xo = x1 + buf * STEP, wx = w0 + nb * STEP, xx = x0 + nb * STEP;
            bind(a[0], b[0]);
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const int n = i * TM + j;
                    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[0][i]), "v"(b[0][j]));
                    if (n % S == S - 1 && n / S < NF) read(n / S, wo, xo, a[1], b[1]);
                }
            bind(a[1], b[1]);                                       // this wave's reads of the buffer are done
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * NQ) : "memory");        // its part of the next k-step has landed
            __builtin_amdgcn_s_barrier();                           // everybody's
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const int n = i * TM + j;
                    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[1][i]), "v"(b[1][j]));
                    if (n % S == S - 1 && n / S < NF) { read(n / S, wx, xx, a[0], b[0]); stage1(buf, kn, n / S); }
                }
            buf = nb;
        };
        for (;;) {
            asm volatile("s_nop 7" ::: "memory");                   // (cleared accumulators: written by the VALU, next read by an MFMA that the compiler does not see)
#pragma unroll 1
            for (int ks = NBUF; ks < KS; ++ks) step(ks);
            const bool more = t + stride < tiles;                   // the last NBUF steps request the next tile's first ones (or their own last one again, never read)
            if (more) point(t + stride);
#pragma unroll 1
            for (int i = 0; i < NBUF; ++i) step(more ? i : KS - 1);
            bind(a[0], b[0]);
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");         // (the last products are in their registers before anything reads them)
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) asm volatile("" : "+a"(acc[i][j]));      // (nor may a copy of an accumulator stand in front of that wait)
            epi(t, acc);
            if (!more) break;
            t += stride;
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // (no DMA into the LDS of a block that has ended)
    }
};
