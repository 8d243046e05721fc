// whisper_kernels.hip - Whisper encoder kernels (compute-bound side of the STT path) for gfx950.
//
// Reference being replaced: WhisperEncoder / WhisperEncoderLayer / WhisperAttention
// (Sources/MLXAudioSTT/Models/Whisper/WhisperLayers.swift:11-156) whose arithmetic is MLX (Conv1d, Linear,
// LayerNorm, gelu, MLXFast.scaledDotProductAttention).  The decoder's per-token path reuses the
// weight-streaming kernels of lm_kernels.hip.  bf16 storage, f32 accumulation, rounding at every MLX
// primitive boundary (oracle/whisper.py).
//
//   k_gemm_big      C[M][N] = X[M][K] W[N][K]^T on v_mfma_f32_16x16x32_bf16, 128x128x32 LDS tiles, fused
//                   bias / exact-erf GELU / residual / positional-embedding epilogues (M = batch*1500 rows)
//   k_layernorm     row LayerNorm (f32 statistics)
//   k_im2col3       k=3 convolution patches (stride 1 / 2) so both stem convs run on k_gemm_big
//   k_scatter_kv    [M][*] K and V columns -> the tiled MFMA-fragment cache layouts of lm_kernels.hip
//   k_attn_prefill  non-causal flash attention over the tiled K/V, 16 query rows per wave
#include "common.h"
#include "gemm_tiles.h"
#include "whisper_kernels.h"
#include <type_traits>

// GELU (erf form, WhisperLayers.swift:142-156 via MLXNN.GELU) for the encoder's big-GEMM epilogues.  erff() from the device library is
// ~60 instructions per element once both of its range branches run in a wave - 15 us per 256 x 256 output tile, fully exposed with one
// block per CU (k_gemm_big3<GELU> 237.7 us against 187.6 us for the same main loop without epilogue, profiles/r04/c6_whisper_kernel_stats.csv).
// Here: erfc(|z|) = poly5(t) exp(-z^2), t = 1 / (1 + 0.3275911 |z|) (Abramowitz & Stegun 7.1.26, |error| <= 1.5e-7), branch-free, and
// 1 + erf(z) taken as erfc(-z) for z < 0 - no cancellation on the negative side.  Against the float64 value, after the bf16 rounding
// that follows: max |diff| 1.0e-6 of full scale, fewer mismatching roundings than the float32 0.5 x (1 + erf) form itself has.
// 1 / d to the nearest float for 1 <= d < 2^14: the hardware reciprocal (1 ulp) and one Newton step, three instructions where the division takes ten.  Equal to the
// division for each of the 117 M values (mis_debug_gelu_rcp_misses counts them; the reciprocal alone misses 12.6 M).
__device__ __forceinline__ float rcp_nearest(float d) {
    const float t = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, t, 1.0f), t, t);
}
__device__ __forceinline__ float gelu_erfc_w(float x) {                   // erfc(|x| / sqrt 2)
    const float z = fminf(fabsf(x) * 0.70710678118654752f, 16.0f);      // (exp(-z^2) is 0 from 10.2 on)
    const float t = rcp_nearest(1.0f + 0.3275911f * z);
    float p = 1.061405429f;
    p = p * t - 1.453152027f;
    p = p * t + 1.421413741f;
    p = p * t - 0.284496736f;
    p = p * t + 0.254829592f;
    return p * t * __expf(-(z * z));
}
__device__ __forceinline__ float gelu_erf_w(float x) {
    const float ec = gelu_erfc_w(x);
    return 0.5f * x * (x >= 0.0f ? 2.0f - ec : ec);
}

__global__ void k_rcp_misses(uint32_t lo, uint32_t n, unsigned long long* misses) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const float d = __uint_as_float(lo + min(i, n - 1));
    if (i < n && rcp_nearest(d) != 1.0f / d) atomicAdd(misses, 1ull);
}
extern "C" mis_status mis_debug_gelu_rcp_misses(int device, int64_t* misses) {
    MIS_API_BEGIN
    MIS_REQUIRE(misses, MIS_ERR_INVALID_INPUT, "null argument");
    HIP_CHECK(hipSetDevice(device));
    const uint32_t lo = 0x3f800000u, n = 0x46800000u - lo;                // 1.0f, 2^14
    DevBuf<unsigned long long> c;
    c.alloc(1);
    HIP_CHECK(hipMemset(c.p, 0, 8));
    hipLaunchKernelGGL(k_rcp_misses, dim3((n + 255) / 256), dim3(256), 0, 0, lo, n, c.p);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpy(misses, c.p, 8, hipMemcpyDeviceToHost));
    MIS_API_END
}

// ============================================================================ big GEMM
#define BG_BM 128
#define BG_BN 128
#define BG_BK 32
#define BG_LD 40          // padded LDS row (bf16 elements): 80 B rows keep 16-B fragments aligned

template <int EPI>
__global__ void __launch_bounds__(256) k_gemm_big(BigGemmParams p) {
    __shared__ __attribute__((aligned(16))) bf16_t Ws[BG_BN][BG_LD];
    __shared__ __attribute__((aligned(16))) bf16_t Xs[BG_BM][BG_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * BG_BN, m0 = blockIdx.y * BG_BM;
    const int wn = wave >> 1, wm = wave & 1;            // wave tile: 64 n x 64 m
    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // staging: 128 rows x 32 k = 512 chunks of 16 B per operand, two per thread
    const int r0 = tid >> 2, c0 = (tid & 3) * 8;
    uint4 wreg[2], xreg[2];
    auto load = [&](int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int row = r0 + 64 * h;
            int n = n0 + row, m = m0 + row;
            wreg[h] = (n < p.N) ? *reinterpret_cast<const uint4*>(p.W + (size_t)n * p.K + k0 + c0) : make_uint4(0, 0, 0, 0);
            xreg[h] = (m < p.M) ? *reinterpret_cast<const uint4*>(p.X + (size_t)m * p.ldx + k0 + c0) : make_uint4(0, 0, 0, 0);
        }
    };
    load(0);
    for (int k0 = 0; k0 < p.K; k0 += BG_BK) {
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<uint4*>(&Ws[r0 + 64 * h][c0]) = wreg[h];
            *reinterpret_cast<uint4*>(&Xs[r0 + 64 * h][c0]) = xreg[h];
        }
        __syncthreads();
        if (k0 + BG_BK < p.K) load(k0 + BG_BK);
        bf16x8_t a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[i] = *reinterpret_cast<const bf16x8_t*>(&Ws[wn * 64 + i * 16 + (lane & 15)][(lane >> 4) * 8]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            b[j] = *reinterpret_cast<const bf16x8_t*>(&Xs[wm * 64 + j * 16 + (lane & 15)][(lane >> 4) * 8]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    // epilogue: C/D lane l, reg r: n = (l>>4)*4 + r (A rows), m = l&15 (B cols) -> 4 consecutive n per lane
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int n = n0 + wn * 64 + i * 16 + (lane >> 4) * 4;
        if (n >= p.N) continue;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[e] = (n + e < p.N) ? bf16_to_f32(p.bias[n + e]) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int m = m0 + wm * 64 + j * 16 + (lane & 15);
            if (m >= p.M) continue;
            uint16_t res[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = bf16_round_f32(acc[i][j][e] + bv[e]);                       // T(xW^T + b)
                if (EPI == BG_GELU || EPI == BG_GELU_POS) v = bf16_round_f32(gelu_erf_w(v));
                if (EPI == BG_RESID) v = bf16_round_f32(v + bf16_to_f32(p.R[(size_t)m * p.N + n + e]));
                if (EPI == BG_GELU_POS) v = bf16_round_f32(v + bf16_to_f32(p.R[(size_t)(m % p.pos_rows) * p.N + n + e]));
                res[e] = f32_to_bf16(v);
            }
            bf16_t* o = p.C + (size_t)m * p.N + n;
            if (n + 3 < p.N) {
                uint2 v;
                v.x = (uint32_t)res[0] | ((uint32_t)res[1] << 16);
                v.y = (uint32_t)res[2] | ((uint32_t)res[3] << 16);
                *reinterpret_cast<uint2*>(o) = v;
            } else {
                for (int e = 0; e < 4 && n + e < p.N; ++e) o[e] = res[e];
            }
        }
    }
}

// ---- the same contraction with direct global -> LDS staging (global_load_lds_dwordx4), BK = 64, two LDS buffers, ONE barrier per
// k-step: tile kt+1 is in flight while the 32 MFMAs per wave of tile kt run.  A wave's LDS-DMA writes 64 lanes x 16 B = 1 KiB
// contiguously (lane-linear destination), i.e. 8 rows x 128 B of the [128][64] bf16 tile; bank conflicts of the fragment reads are
// avoided on the SOURCE side: LDS position (row r, 16-B chunk c) holds global chunk c ^ ((r >> 1) & 7), and a fragment read of
// chunk kc of row r goes to position kc ^ ((r >> 1) & 7).  With ds_read_b128's 16-lane service groups ({0-3,12-15,20-27}, ...: every
// group touches the 16 rows of a fragment once, at two neighbouring kc) the 16 lanes of a group land on 16 distinct 16-B slots of
// the 256-B bank row.  Rows past M / N are loaded clamped and masked in the epilogue.
#define BG2_BK 64
template <int EPI>
__global__ void __launch_bounds__(256, 2) k_gemm_big2(BigGemmParams p) {
    __shared__ __attribute__((aligned(1024))) bf16_t Ws[2][BG_BN * BG2_BK];
    __shared__ __attribute__((aligned(1024))) bf16_t Xs[2][BG_BM * BG2_BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * BG_BN, m0 = blockIdx.y * BG_BM;
    const int wn = wave >> 1, wm = wave & 1;            // wave tile: 64 n x 64 m
    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // staging: instruction q (0..3) of wave w moves rows (w*4 + q)*8 .. +8 of each operand tile; lane l -> row + (l >> 3), position l & 7
    const bf16_t* wsrc[4];
    const bf16_t* xsrc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = (wave * 4 + q) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        const int n = min(n0 + r, p.N - 1), m = min(m0 + r, p.M - 1);
        wsrc[q] = p.W + (size_t)n * p.K + chunk * 8;
        xsrc[q] = p.X + (size_t)m * p.ldx + chunk * 8;
    }
    auto stage = [&](int buf, int k0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row0 = (wave * 4 + q) * 8;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wsrc[q] + k0),
                                             (__attribute__((address_space(3))) void*)&Ws[buf][row0 * BG2_BK], 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xsrc[q] + k0),
                                             (__attribute__((address_space(3))) void*)&Xs[buf][row0 * BG2_BK], 16, 0, 0);
        }
    };
    const int sw = (lane >> 1) & 7;                      // ((row >> 1) & 7) of this lane's fragment rows (row = 16*t + (lane & 15))
    const int KT = p.K / BG2_BK;
    stage(0, 0);
    for (int kt = 0; kt < KT; ++kt) {
        __syncthreads();                                 // waits for this wave's LDS-DMA (vmcnt(0)), then the block: tile kt is complete
        const bf16_t* wt = Ws[kt & 1];
        const bf16_t* xt = Xs[kt & 1];
        // all fragment reads of the tile FIRST, then the next tile's DMA: hipcc puts a vmcnt(0) in front of any ds_read that follows an
        // LDS-DMA in program order (it cannot prove the read does not alias the DMA's destination), which would serialise the
        // prefetch with the reads; issued after them, the DMA runs under the 32 MFMAs of this tile
        bf16x8_t a[2][4], b[2][4];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int pos = ((ks * 4 + (lane >> 4)) ^ sw) * 8;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                a[ks][i] = *reinterpret_cast<const bf16x8_t*>(wt + (wn * 64 + i * 16 + (lane & 15)) * BG2_BK + pos);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b[ks][j] = *reinterpret_cast<const bf16x8_t*>(xt + (wm * 64 + j * 16 + (lane & 15)) * BG2_BK + pos);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < KT) stage((kt + 1) & 1, (kt + 1) * BG2_BK);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
    }
    // epilogue: as k_gemm_big
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int n = n0 + wn * 64 + i * 16 + (lane >> 4) * 4;
        if (n >= p.N) continue;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[e] = (n + e < p.N) ? bf16_to_f32(p.bias[n + e]) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int m = m0 + wm * 64 + j * 16 + (lane & 15);
            if (m >= p.M) continue;
            uint16_t res[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = bf16_round_f32(acc[i][j][e] + bv[e]);                       // T(xW^T + b)
                if (EPI == BG_GELU || EPI == BG_GELU_POS) v = bf16_round_f32(gelu_erf_w(v));
                if (EPI == BG_RESID) v = bf16_round_f32(v + bf16_to_f32(p.R[(size_t)m * p.N + n + e]));
                if (EPI == BG_GELU_POS) v = bf16_round_f32(v + bf16_to_f32(p.R[(size_t)(m % p.pos_rows) * p.N + n + e]));
                res[e] = f32_to_bf16(v);
            }
            bf16_t* o = p.C + (size_t)m * p.N + n;
            if (n + 3 < p.N) {
                uint2 v;
                v.x = (uint32_t)res[0] | ((uint32_t)res[1] << 16);
                v.y = (uint32_t)res[2] | ((uint32_t)res[3] << 16);
                *reinterpret_cast<uint2*>(o) = v;
            } else {
                for (int e = 0; e < 4 && n + e < p.N; ++e) o[e] = res[e];
            }
        }
    }
}

// ---------------------------------------------------------------------------- 256 x 256 tiles, eight waves, counted waits
// Round 4 (tools/gemm_lab/big_lab, profiles/r04/big_lab.jsonl): at the encoder's shapes (M = 8 x 1500 rows, N, K in 1280 .. 5120) a
// 256 x 256 x 64 tile on eight waves - one block per CU, two 64 KB LDS buffers - runs the four GEMMs of a layer in 135.7 / 44.6 / 187.6 /
// 158.4 us against 151.2 / 52.0 / 203.9 / 181.5 for k_gemm_big2 (35-40 % of the dense bf16 MFMA peak instead of 31-35 %): each wave's
// fragment reads feed twice the MFMAs (44 FLOP per LDS byte against 32).  The deeper rings of the same laboratory (three buffers at
// 256 x 128 / 128 x 256) were slower.  What makes the two-buffer form work is WHEN the waves wait: the LDS-DMA of tile kt + 1 is issued
// behind the fragment reads of tile kt and waited for with an explicit vmcnt(0) right in front of the next raw s_barrier - with compiler
// loads hipcc puts a vmcnt(0) in front of every ds_read that follows an LDS-DMA in program order, hence asm reads (ds_read_b128, one
// lgkmcnt(0) naming every fragment in front of the MFMAs).  Same k order and accumulators as k_gemm_big2: bit-identical C.
__device__ __forceinline__ uint32_t bg3_lds_offset(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
__device__ __forceinline__ bf16x8_t bg3_lds_read16(uint32_t addr) {
    bf16x8_t v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr) : "memory");
    return v;
}
#define BG3_BM 256
#define BG3_BN 256
template <int EPI, int WM, int WN>
__device__ __forceinline__ void gemm_big3_body(const BigGemmParams& p) {
    constexpr int NW = WM * WN;                                  // 8 waves
    constexpr int TM = BG3_BM / WM / 16, TN = BG3_BN / WN / 16;  // 16 x 16 MFMA tiles per wave (m, n)
    constexpr int QW = BG3_BN / 8 / NW, QX = BG3_BM / 8 / NW;    // LDS-DMA instructions per wave and tile (8 rows of 128 B each)
    static_assert(NW == 8, "eight waves");
    extern __shared__ __attribute__((aligned(1024))) bf16_t bg3_lds[];
    bf16_t* Ws = bg3_lds;                                        // [2][BN * 64]
    bf16_t* Xs = bg3_lds + (size_t)2 * BG3_BN * BG2_BK;          // [2][BM * 64]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Blocks are dealt to the XCDs by id mod 8.  Up to 8 column tiles an XCD takes a contiguous range of row tiles and walks it column tile by column tile:
    // the blocks it runs together share 6 tiles of X and 5 of W in one L2 (fc2 169 -> 158 us, out_proj 62 -> 58); with more column tiles the row-major
    // order is the faster one (q|k|v 135 against 143 us).
    const int nt = (p.N + BG3_BN - 1) / BG3_BN, mt = (p.M + BG3_BM - 1) / BG3_BM;
    int ni = blockIdx.x % nt, mi = blockIdx.x / nt;
    if (nt <= 8) {
        const int xcd = blockIdx.x & 7, j0 = blockIdx.x >> 3, mlo = mt * xcd / 8, mcnt = mt * (xcd + 1) / 8 - mlo;
        if (j0 >= mcnt * nt) return;
        ni = j0 / mcnt; mi = mlo + j0 % mcnt;
    }
    const int n0 = ni * BG3_BN, m0 = mi * BG3_BM;
    const int wn = wave / WM, wm = wave % WM;
    // Value tiles of BG_KV swap the operands: a lane then holds four consecutive KEYS of one dim, which are one 8-byte piece of the value image (two bytes each
    // the other way round).  The tile is square, so only the sources and the epilogue differ; the products and their order do not.
    // (k_gemm_kv_tiles, 8 windows: q|k|v 134 us, cross k|v 86 us, where GEMM and scatter kernel took 139 + 20 and 89 + 20)
    const bool swp = EPI == BG_KV && n0 >= p.vcol0;
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const bf16_t* wsrc[QW];
    const bf16_t* xsrc[QX];
#pragma unroll
    for (int q = 0; q < QW; ++q) {
        const int r = (wave * QW + q) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        wsrc[q] = swp ? p.X + (size_t)min(m0 + r, p.M - 1) * p.ldx + chunk * 8 : p.W + (size_t)min(n0 + r, p.N - 1) * p.K + chunk * 8;
    }
#pragma unroll
    for (int q = 0; q < QX; ++q) {
        const int r = (wave * QX + q) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        xsrc[q] = swp ? p.W + (size_t)min(n0 + r, p.N - 1) * p.K + chunk * 8 : p.X + (size_t)min(m0 + r, p.M - 1) * p.ldx + chunk * 8;
    }
    auto stage = [&](int buf, int k0) {
#pragma unroll
        for (int q = 0; q < QW; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wsrc[q] + k0),
                                             (__attribute__((address_space(3))) void*)&Ws[((size_t)buf * BG3_BN + (wave * QW + q) * 8) * BG2_BK], 16, 0, 0);
#pragma unroll
        for (int q = 0; q < QX; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xsrc[q] + k0),
                                             (__attribute__((address_space(3))) void*)&Xs[((size_t)buf * BG3_BM + (wave * QX + q) * 8) * BG2_BK], 16, 0, 0);
    };
    const int KT = p.K / BG2_BK;
    const int sw = (lane >> 1) & 7;
    const uint32_t ws_base = bg3_lds_offset(Ws) + (uint32_t)((wn * (BG3_BN / WN) + (lane & 15)) * BG2_BK * 2);
    const uint32_t xs_base = bg3_lds_offset(Xs) + (uint32_t)((wm * (BG3_BM / WM) + (lane & 15)) * BG2_BK * 2);
    stage(0, 0);
    for (int kt = 0; kt < KT; ++kt) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // this wave's part of tile kt has landed
        __builtin_amdgcn_s_barrier();                            // every wave's part is in LDS; the other buffer is free
        asm volatile("" ::: "memory");
        const int buf = kt & 1;
        bf16x8_t a[2][TN], b[2][TM];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const uint32_t pos = (uint32_t)(((ks * 4 + (lane >> 4)) ^ sw) * 16);
#pragma unroll
            for (int i = 0; i < TN; ++i) a[ks][i] = bg3_lds_read16(ws_base + (uint32_t)((buf * BG3_BN + i * 16) * BG2_BK * 2) + pos);
#pragma unroll
            for (int j = 0; j < TM; ++j) b[ks][j] = bg3_lds_read16(xs_base + (uint32_t)((buf * BG3_BM + j * 16) * BG2_BK * 2) + pos);
        }
        // the next DMA goes into the buffer read one k-step ago; issued behind this tile's reads, it runs under its MFMAs
        if (kt + 1 < KT) stage((kt + 1) & 1, (kt + 1) * BG2_BK);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            // one wait, naming every fragment of this half; the other half's reads (LDS returns in order) run under its MFMAs
            if (ks == 0) asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(a[0][0]) : "n"(TN + TM));
            else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[1][0]));
#pragma unroll
            for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(a[ks][i]));
#pragma unroll
            for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(b[ks][j]));
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
        }
    }
    if constexpr (EPI == BG_KV) {
        auto pack4 = [](const f32x4_t& v, float b0, float b1, float b2, float b3) {
            uint2 o;
            o.x = (uint32_t)f32_to_bf16(v[0] + b0) | ((uint32_t)f32_to_bf16(v[1] + b1) << 16);
            o.y = (uint32_t)f32_to_bf16(v[2] + b2) | ((uint32_t)f32_to_bf16(v[3] + b3) << 16);
            return o;
        };
        if (swp) {                                       // rows of the tile: keys; lane & 15: dim.  Image [D/16][64 lanes][8]: lane (key / 8) 16 + d & 15, key & 7
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int m = m0 + wn * (BG3_BN / WN) + i * 16 + (lane >> 4) * 4;
                if (m >= p.M) continue;                  // (M and T are multiples of 4: four keys share a batch row and a piece)
                const int br = m / p.T, t = m - br * p.T, pr = t & 31;
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const int dd = n0 - p.vcol0 + wm * (BG3_BM / WM) + j * 16 + (lane & 15), hd = dd >> 6, d = dd & 63;
                    const float bv = p.bias ? bf16_to_f32(p.bias[p.vcol0 + dd]) : 0.0f;
                    bf16_t* o = p.vc + (((size_t)br * p.H + hd) * p.Spad + (t & ~31)) * 64 + (d >> 4) * 512 + ((pr >> 3) * 16 + (d & 15)) * 8 + (pr & 7);
                    *reinterpret_cast<uint2*>(o) = pack4(acc[i][j], bv, bv, bv, bv);
                }
            }
            return;
        }
        if (n0 >= p.kcol0) {                             // image [2][D/32][64 lanes][8]: the key permutation of k_scatter_kv
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int m = m0 + wm * (BG3_BM / WM) + j * 16 + (lane & 15);
                if (m >= p.M) continue;
                const int br = m / p.T, t = m - br * p.T, pr = t & 31, prow = ((pr >> 3) << 2) | (pr & 3), half = (pr >> 2) & 1;
#pragma unroll
                for (int i = 0; i < TN; ++i) {
                    const int dd = n0 - p.kcol0 + wn * (BG3_BN / WN) + i * 16 + (lane >> 4) * 4, hd = dd >> 6, d = dd & 63;
                    float bv[4] = {0.f, 0.f, 0.f, 0.f};
                    if (p.bias) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) bv[e] = bf16_to_f32(p.bias[p.kcol0 + dd + e]);
                    }
                    bf16_t* o = p.kc + (((size_t)br * p.H + hd) * p.Spad + (t & ~31)) * 64 + (half * 2 + (d >> 5)) * 512 + (((d & 31) >> 3) * 16 + prow) * 8 + (d & 7);
                    *reinterpret_cast<uint2*>(o) = pack4(acc[i][j], bv[0], bv[1], bv[2], bv[3]);
                }
            }
            return;
        }
    }
    // epilogue: as k_gemm_big2 (C/D lane = column m (l & 15), rows n = 4 (l >> 4) + e)
#pragma unroll
    for (int i = 0; i < TN; ++i) {
        const int n = n0 + wn * (BG3_BN / WN) + i * 16 + (lane >> 4) * 4;
        if (n >= p.N) continue;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[e] = (n + e < p.N) ? bf16_to_f32(p.bias[n + e]) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int m = m0 + wm * (BG3_BM / WM) + j * 16 + (lane & 15);
            if (m >= p.M) continue;
            uint16_t res[4];
            float rv[4] = {0.f, 0.f, 0.f, 0.f};                                     // residual / positional row: ONE 8-byte load (N % 4 == 0)
            if (EPI == BG_RESID || EPI == BG_GELU_POS) {
                const size_t rrow = EPI == BG_RESID ? (size_t)m : (size_t)(m % p.pos_rows);
                const uint2 rq = *reinterpret_cast<const uint2*>(p.R + rrow * p.N + n);
                rv[0] = __uint_as_float(rq.x << 16); rv[1] = __uint_as_float(rq.x & 0xffff0000u);
                rv[2] = __uint_as_float(rq.y << 16); rv[3] = __uint_as_float(rq.y & 0xffff0000u);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = bf16_round_f32(acc[i][j][e] + bv[e]);                       // T(xW^T + b)
                if (EPI == BG_GELU || EPI == BG_GELU_POS) v = bf16_round_f32(gelu_erf_w(v));
                if (EPI == BG_RESID || EPI == BG_GELU_POS) v = bf16_round_f32(v + rv[e]);
                res[e] = f32_to_bf16(v);
            }
            bf16_t* o = p.C + (size_t)m * p.N + n;
            uint2 v;
            v.x = (uint32_t)res[0] | ((uint32_t)res[1] << 16);
            v.y = (uint32_t)res[2] | ((uint32_t)res[3] << 16);
            *reinterpret_cast<uint2*>(o) = v;                                       // (n < N and N % 4 == 0: the four columns exist)
        }
    }
}
template <int EPI, int WM, int WN>
__global__ void __launch_bounds__(512, 1) k_gemm_big3(BigGemmParams p) { gemm_big3_body<EPI, WM, WN>(p); }
template <int WM, int WN>
__global__ void __launch_bounds__(512, 1) k_gemm_kv_tiles(BigGemmParams p) { gemm_big3_body<BG_KV, WM, WN>(p); }
template <int EPI, int WM, int WN>
static bool launch_big3_one(const BigGemmParams& p, hipStream_t s) {
    constexpr int lds_bytes = 2 * (BG3_BM + BG3_BN) * BG2_BK * 2;            // 128 KB
    void (*kernel)(BigGemmParams);
    if constexpr (EPI == BG_KV) kernel = k_gemm_kv_tiles<WM, WN>;
    else kernel = k_gemm_big3<EPI, WM, WN>;
    static const bool ok = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) == hipSuccess;
    if (!ok) { (void)hipGetLastError(); return false; }
    const int nt = cdiv(p.N, BG3_BN), mt = cdiv(p.M, BG3_BM);
    hipLaunchKernelGGL(kernel, dim3(nt <= 8 ? 8 * nt * cdiv(mt, 8) : nt * mt), dim3(512), lds_bytes, s, p);
    return true;
}
template <int EPI>
static bool launch_big3(const BigGemmParams& p, hipStream_t s) {
    // wave grid as measured: 2 (m) x 4 (n) for the wide / deep MLP shapes, 4 x 2 otherwise
    return (p.N >= 4096 || p.K >= 4096) ? launch_big3_one<EPI, 2, 4>(p, s) : launch_big3_one<EPI, 4, 2>(p, s);
}

// ---------------------------------------------------------------------------- tiles of 32 TM x 256 outputs, four waves (gemm_tiles.h)
// What it gives over k_gemm_big3 (large-v3, us per launch): 8 x 1500 rows q|k|v 122 / 140, o 55 / 60, fc1 171 / 211, fc2 146 / 172, cross k|v 88 / 101; 6 x 1500
// (k_gemm_big2 where 180 tiles of 256 x 256 were too few) 100 / 128, 44 / 58, 128 / 159, 122 / 173, 66 / 90; 4 x 1500 71 / 89, 33 / 34, 93 / 107, 85 / 95, 45 / 50.
// k_gemm_big3 keeps K = 128 (the ring takes three k-steps) and operands past 32-bit offsets; no size of the family has either.
// TM by the rounds of 256 persistent blocks it makes (launch_gemm_rows).  Products in the order of k: the bits of k_gemm_big2.
// A GELU after T(xW^T + b) is a function of sixteen bits: gelu_erf_w(v) = v f(v), f in an LDS table over |v| = 2^-10 .. 16 and the sign (14 KB; below 2^-10 the
// result is v / 2, exact from 2^-125 on, above 16 it is v or -0: the values that the clamped factors round to).  The same bits as the formula, in 12 instructions an
// output and an LDS read for 31, two of them of quarter rate - a block's only waves wait for them.  fc1, eight windows 204 -> 171 us, one 31 -> 28.
struct GeluTable {
    static constexpr uint32_t LO = 0x3a80, HI = 0x4180, N = HI - LO + 1;           // bf16 of 2^-10 and 16
    static __device__ __forceinline__ void fill(float* tab) {                      // (ends with a barrier)
        for (uint32_t i = threadIdx.x; i < N; i += 256) {
            const float z = __uint_as_float((LO + i) << 16), ec = gelu_erfc_w(z);
            tab[i] = 0.5f * (2.0f - ec);
            tab[N + i] = 0.5f * ec;
        }
        __syncthreads();
    }
    // x[e] = gelu(x[e]) before its rounding; x of 16 bits.  base: LDS offset of the table
    static __device__ __forceinline__ void apply(uint32_t base, float (&x)[16]) {
        uint32_t a[16];
        float f[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float y = __builtin_amdgcn_fmed3f(fabsf(x[e]), __uint_as_float(LO << 16), __uint_as_float(HI << 16));
            a[e] = (__float_as_uint(y) >> 14) + ((uint32_t)((int)__float_as_uint(x[e]) >> 31) & (4 * N)) + (base - 4 * LO);
        }
        // (reads and their wait in one block: behind an LDS-DMA the compiler would wait for every load and store in flight)
        asm volatile("ds_read_b32 %0, %16\n\tds_read_b32 %1, %17\n\tds_read_b32 %2, %18\n\tds_read_b32 %3, %19\n\t"
                     "ds_read_b32 %4, %20\n\tds_read_b32 %5, %21\n\tds_read_b32 %6, %22\n\tds_read_b32 %7, %23\n\t"
                     "ds_read_b32 %8, %24\n\tds_read_b32 %9, %25\n\tds_read_b32 %10, %26\n\tds_read_b32 %11, %27\n\t"
                     "ds_read_b32 %12, %28\n\tds_read_b32 %13, %29\n\tds_read_b32 %14, %30\n\tds_read_b32 %15, %31\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]), "=&v"(f[6]), "=&v"(f[7]),
                       "=&v"(f[8]), "=&v"(f[9]), "=&v"(f[10]), "=&v"(f[11]), "=&v"(f[12]), "=&v"(f[13]), "=&v"(f[14]), "=&v"(f[15])
                     : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
                       "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]), "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15])
                     : "memory");
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] *= f[e];
    }
};
template <int EPI, int TM>
__device__ __forceinline__ void gemm_rows_body(const BigGemmParams& p) {
    using T = GemmTiles<TM, false>;
    constexpr int G = TM >= 6 ? 6 : 8;
    constexpr bool GELU = EPI == BG_GELU || EPI == BG_GELU_POS;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[T::LDS];
    __shared__ float gelu_tab[GELU ? 2 * GeluTable::N : 1];
    // Value tiles of BG_KV swap the operands: a lane then holds four consecutive KEYS of one dim, which are one 8-byte piece of the value image (two bytes each
    // the other way round).  They are numbered behind the others, 256 keys x 32 TM dims each; the products and their order are the same.
    const int N0 = EPI == BG_KV ? p.vcol0 : p.N;
    const TileOrder o0{(p.M + T::BM - 1) / T::BM, (N0 + T::BN - 1) / T::BN}, o1{(p.M + T::BN - 1) / T::BN, EPI == BG_KV ? (p.N - N0 + T::BM - 1) / T::BM : 0};
    const int tiles0 = o0.mt * o0.nt, tiles = tiles0 + o1.mt * o1.nt;
    const int xcd = blockIdx.x & 7, lo = (int)((int64_t)tiles * xcd / 8), hi = (int)((int64_t)tiles * (xcd + 1) / 8), first = lo + (blockIdx.x >> 3);
    if (first >= hi) return;
    if constexpr (GELU) GeluTable::fill(gelu_tab);
    auto where = [&](int t, bool& swp, int& m0, int& n0) {
        int mi, ni;
        swp = EPI == BG_KV && t >= tiles0;
        if (swp) { o1.at(G, t - tiles0, mi, ni); m0 = mi * T::BN; n0 = N0 + ni * T::BM; }
        else { o0.at(G, t, mi, ni); m0 = mi * T::BM; n0 = ni * T::BN; }
    };
    bool sw; int mt0, nt0;                                   // of the tile being requested
    T::run(lds, p.K, first, gridDim.x >> 3, hi,
           [&](int t, const bf16_t*& Wb, const bf16_t*& Xb) {
               where(t, sw, mt0, nt0);
               Wb = sw ? p.X : p.W;
               Xb = sw ? p.W : p.X;
           },
           [&](int, int q, int lane) {
               const int r = q * 8 + (lane >> 3);
               return (sw ? (uint32_t)min(mt0 + r, p.M - 1) * p.ldx : (uint32_t)min(nt0 + r, N0 - 1) * p.K) + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
           },
           [&](int, int r) { return sw ? (uint32_t)min(nt0 + r, p.N - 1) * p.K : (uint32_t)min(mt0 + r, p.M - 1) * p.ldx; },
           [&](int t, const f32x4_t (&acc)[T::TN][TM]) {
               bool swp; int m0, n0;
               where(t, swp, m0, n0);
               int lane = threadIdx.x & 63;
               asm volatile("" : "+v"(lane));
               const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = (wave >> 1) * 128 + (lane >> 4) * 4, xr = (wave & 1) * TM * 16 + (lane & 15);
               auto pack4 = [](float a, float b, float c, float d) {
                   typedef float f2_t __attribute__((ext_vector_type(2)));
                   typedef __bf16 h2_t __attribute__((ext_vector_type(2)));
                   return make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){a, b}, h2_t)), __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){c, d}, h2_t)));
               };
               auto part = [](const uint2& b, int e) { return __uint_as_float(e & 1 ? (e < 2 ? b.x : b.y) & 0xffff0000u : (e < 2 ? b.x : b.y) << 16); };
               uint2 bv[T::TN];
#pragma unroll
               for (int i = 0; i < T::TN; ++i) bv[i] = p.bias ? *reinterpret_cast<const uint2*>(p.bias + min(n0 + wr + i * 16, N0 - 4)) : make_uint2(0, 0);
               if constexpr (EPI == BG_KV) {
                   // an output's byte offset is the sum of one of its W row and one of its X row, in C, in the key image [2][D/32][64 lanes][8] (the key permutation
                   // of k_scatter_kv) and in the value image [D/16][64 lanes][8] (lane (key / 8) 16 + d & 15, key & 7); one loop for the three
                   const bool key = !swp && n0 >= p.kcol0;
                   unsigned char* const base = reinterpret_cast<unsigned char*>(swp ? p.vc : key ? p.kc : p.C);
                   auto of_key = [&](int m) {                // (M and T are multiples of 4: four keys share a batch row and a piece)
                       const uint32_t br = (uint32_t)m / (uint32_t)p.T, tk = m - br * p.T, pr = tk & 31;
                       return br * p.H * p.Spad * 128u + (tk & ~31u) * 128u + (swp ? (pr >> 3) * 256 + (pr & 7) * 2 : ((pr >> 2) & 1) * 2048 + (((pr >> 3) << 2) | (pr & 3)) * 16);
                   };
                   auto of_dim = [&](int dd) {
                       const uint32_t d = dd & 63;
                       return (uint32_t)(dd >> 6) * p.Spad * 128u + (swp ? (d >> 4) * 1024 + (d & 15) * 16 : ((d >> 5) * 512 + ((d & 31) >> 3) * 128 + (d & 7)) * 2);
                   };
                   uint32_t at[T::TN];
                   bool ok[T::TN];
#pragma unroll
                   for (int i = 0; i < T::TN; ++i) {
                       ok[i] = !swp || m0 + wr + i * 16 < p.M;
                       at[i] = swp ? of_key(m0 + wr + i * 16) : key ? of_dim(n0 - p.kcol0 + wr + i * 16) : (uint32_t)(n0 + wr + i * 16) * 2;
                       if (swp) bv[i] = make_uint2(0, 0);
                   }
#pragma unroll
                   for (int j = 0; j < TM; ++j) {
                       __builtin_amdgcn_sched_barrier(0);
                       const int x = (swp ? n0 : m0) + xr + j * 16, xn = swp ? min(x, p.N - 1) : 0;
                       const float b = swp && p.bias ? bf16_to_f32(p.bias[xn]) : 0.0f;
                       const bool okx = x < (swp ? p.N : p.M);
                       const uint32_t to = swp ? of_dim(xn - N0) : key ? of_key(x) : (uint32_t)x * p.N * 2u;
#pragma unroll
                       for (int i = 0; i < T::TN; ++i) {
                           float v[4];
#pragma unroll
                           for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + part(bv[i], e) + b;
                           const uint2 o = pack4(v[0], v[1], v[2], v[3]);
                           if (okx & ok[i]) *reinterpret_cast<uint2*>(base + at[i] + to) = o;
                       }
                   }
                   return;
               }
               // residual or positional values are requested eight outputs ahead; an output is packed before the branch of its store (a load consumed inside it
               // waits for every store before it)
               constexpr bool RES = EPI == BG_RESID || EPI == BG_GELU_POS;
               uint2 r[T::TN];
               auto residual = [&](int j, int i) {
                   const int m = min(m0 + xr + j * 16, p.M - 1);
                   r[i] = *reinterpret_cast<const uint2*>(reinterpret_cast<const unsigned char*>(p.R) + (uint32_t)(EPI == BG_RESID ? m : m % p.pos_rows) * p.N * 2u + min(n0 + wr + i * 16, p.N - 4) * 2);
               };
               if constexpr (RES) {
#pragma unroll
                   for (int i = 0; i < T::TN; ++i) residual(0, i);
               }
#pragma unroll
               for (int j = 0; j < TM; ++j) {
                   __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                   for (int ih = 0; ih < T::TN; ih += 4) {
                       float v[16];
#pragma unroll
                       for (int e = 0; e < 16; ++e) v[e] = bf16_round_f32(acc[ih + (e >> 2)][j][e & 3] + part(bv[ih + (e >> 2)], e & 3));        // T(xW^T + b)
                       if constexpr (GELU) GeluTable::apply(gt_lds_offset(gelu_tab), v);
#pragma unroll
                       for (int i = ih; i < ih + 4; ++i) {
                           float* w = v + (i - ih) * 4;
                           if constexpr (RES) {
#pragma unroll
                               for (int e = 0; e < 4; ++e) w[e] = (GELU ? bf16_round_f32(w[e]) : w[e]) + part(r[i], e);
                           }
                           uint2 o = pack4(w[0], w[1], w[2], w[3]);
                           asm volatile("" : "+v"(o.x), "+v"(o.y));
                           if constexpr (RES) {
                               if (j + 1 < TM) residual(j + 1, i);
                           }
                           const int m = m0 + xr + j * 16;
                           if (m < p.M && n0 + wr + i * 16 < N0) *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(p.C) + (uint32_t)m * p.N * 2u + (n0 + wr + i * 16) * 2) = o;
                       }
                   }
               }
           });
}
template <int EPI, int TM>
__global__ void __launch_bounds__(256, 1) k_gemm_rows(BigGemmParams p) { gemm_rows_body<EPI, TM>(p); }
template <int TM>
__global__ void __launch_bounds__(256, 1) k_gemm_rows_kv(BigGemmParams p) { gemm_rows_body<BG_KV, TM>(p); }
template <int EPI>
static bool launch_gemm_rows(const BigGemmParams& p, hipStream_t s) {
    // (32-bit byte offsets; three k-steps at least fill the ring)
    if (p.K % BG2_BK || p.K < 3 * BG2_BK || (int64_t)p.N * p.K >= (1ll << 31) || (int64_t)p.M * p.ldx >= (1ll << 31)) return false;
    if ((int64_t)p.M * p.N >= (1ll << 31) || (EPI == BG_KV && (int64_t)(p.M / p.T) * p.H * p.Spad * 128 >= (1ll << 32))) return false;
    const int N0 = EPI == BG_KV ? p.vcol0 : p.N;
    auto count = [&](int tm) { return cdiv(p.M, 32 * tm) * cdiv(N0, 256) + (EPI == BG_KV ? cdiv(p.M, 256) * cdiv(p.N - N0, 32 * tm) : 0); };
    int best = 0;
    double least = 0;
    for (int tm : {8, 6, 5, 4}) {                                  // rounds of 256 blocks, each as long as its tiles are high and a little
        const double cost = cdiv(count(tm), 256) * (tm + 0.4);
        if (tm == 5 && (EPI == BG_GELU || EPI == BG_GELU_POS)) continue;      // (its ring leaves no LDS for the table)
        if (!best || cost < least) { best = tm; least = cost; }
    }
    // fewer tiles leave compute units idle that more blocks of the smaller kernels fill (one window: o 23.9 us there; fc1, 240 tiles: 28 here, 30 there)
    if (count(best) < 200) return false;
    auto go = [&](auto tag) {
        constexpr int TM = decltype(tag)::value;
        void (*kernel)(BigGemmParams);
        if constexpr (EPI == BG_KV) kernel = k_gemm_rows_kv<TM>;
        else kernel = k_gemm_rows<EPI, TM>;
        hipLaunchKernelGGL(kernel, dim3(std::min((int)round_up(count(TM), 8), 256)), dim3(256), 0, s, p);
    };
    if (best == 8) go(std::integral_constant<int, 8>{});
    else if (best == 6) go(std::integral_constant<int, 6>{});
    else if (best == 5) go(std::integral_constant<int, EPI == BG_GELU || EPI == BG_GELU_POS ? 4 : 5>{});
    else go(std::integral_constant<int, 4>{});
    return true;
}

bool launch_gemm_big_kv(const BigGemmParams& p, hipStream_t s) {
    const char* e3 = getenv("MIS_GEMM_BIG3");
    const int mode = e3 ? atoi(e3) : 1;
    // key and value columns start at tile boundaries; pieces of four keys stay inside a batch row
    if (mode == 0 || p.ldx % 8 || p.kcol0 % BG3_BN || p.vcol0 % BG3_BN || p.N % BG3_BN || p.T % 4 || p.M % 4 || p.Spad % 32) return false;
    if (mode == 1 && launch_gemm_rows<BG_KV>(p, s)) return true;
    if (p.K % BG2_BK != 0 || p.K < 2 * BG2_BK || (mode != 2 && (long)cdiv(p.N, BG3_BN) * cdiv(p.M, BG3_BM) < 200)) return false;
    return launch_big3<BG_KV>(p, s);
}

void launch_gemm_big(int epi, const BigGemmParams& p, hipStream_t s) {
    MIS_REQUIRE(p.K % BG_BK == 0 && p.ldx % 8 == 0 && p.N % 4 == 0, MIS_ERR_INVALID_INPUT, "big GEMM needs K %% 32 == 0");
    dim3 grid(cdiv(p.N, BG_BN), cdiv(p.M, BG_BM)), block(256);
    {   // large tiles where their grid still fills most of the chip; below that the 128 x 128 kernel has four times the blocks.
        // MIS_GEMM_BIG3=0: never (A/B); =2: the eight-wave kernel whenever the shape allows (parity tests)
        const char* e3 = getenv("MIS_GEMM_BIG3");
        const int mode = e3 ? atoi(e3) : 1;
        const long blocks3 = (long)cdiv(p.N, BG3_BN) * cdiv(p.M, BG3_BM);
        const bool big3 = p.K % BG2_BK == 0 && p.K >= 2 * BG2_BK && (mode == 2 || blocks3 >= 200);
        auto large = [&](auto tag) {
            constexpr int E = decltype(tag)::value;
            return (mode == 1 && launch_gemm_rows<E>(p, s)) || (mode != 0 && big3 && launch_big3<E>(p, s));
        };
        bool done = false;
        switch (epi) {
            case BG_NONE: done = large(std::integral_constant<int, BG_NONE>{}); break;
            case BG_GELU: done = large(std::integral_constant<int, BG_GELU>{}); break;
            case BG_RESID: done = large(std::integral_constant<int, BG_RESID>{}); break;
            case BG_GELU_POS: done = large(std::integral_constant<int, BG_GELU_POS>{}); break;
            default: throw MisError(MIS_ERR_GENERATION_FAILED, "unknown big GEMM epilogue");
        }
        if (done) return;
    }
    if (p.K % BG2_BK == 0 && p.K >= 2 * BG2_BK) {
        switch (epi) {
            case BG_NONE: hipLaunchKernelGGL((k_gemm_big2<BG_NONE>), grid, block, 0, s, p); return;
            case BG_GELU: hipLaunchKernelGGL((k_gemm_big2<BG_GELU>), grid, block, 0, s, p); return;
            case BG_RESID: hipLaunchKernelGGL((k_gemm_big2<BG_RESID>), grid, block, 0, s, p); return;
            case BG_GELU_POS: hipLaunchKernelGGL((k_gemm_big2<BG_GELU_POS>), grid, block, 0, s, p); return;
            default: throw MisError(MIS_ERR_GENERATION_FAILED, "unknown big GEMM epilogue");
        }
    }
    switch (epi) {
        case BG_NONE: hipLaunchKernelGGL((k_gemm_big<BG_NONE>), grid, block, 0, s, p); break;
        case BG_GELU: hipLaunchKernelGGL((k_gemm_big<BG_GELU>), grid, block, 0, s, p); break;
        case BG_RESID: hipLaunchKernelGGL((k_gemm_big<BG_RESID>), grid, block, 0, s, p); break;
        case BG_GELU_POS: hipLaunchKernelGGL((k_gemm_big<BG_GELU_POS>), grid, block, 0, s, p); break;
        default: throw MisError(MIS_ERR_GENERATION_FAILED, "unknown big GEMM epilogue");
    }
}

// ============================================================================ LayerNorm over rows
__global__ void __launch_bounds__(256) k_layernorm(const bf16_t* __restrict__ x, bf16_t* __restrict__ y,
                                                   const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias, int d,
                                                   float eps) {
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const bf16_t* xr = x + row * d;
    float s = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) s += bf16_to_f32(xr[i]);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)d;
    __syncthreads();
    float q = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) { float t = bf16_to_f32(xr[i]) - mean; q += t * t; }
    q = wave_sum(q);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
    __syncthreads();
    const float rstd = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256)
        y[row * d + i] = f32_to_bf16((bf16_to_f32(xr[i]) - mean) * rstd * bf16_to_f32(w[i]) + bf16_to_f32(bias[i]));
}
// d % 8 == 0, d <= 2048: the row lives in registers (one 16-byte piece per thread, read once), two block sums, 16-byte stores - the
// element-wise kernel above reads the row three times with 2-byte loads (32.6 us per 12 000 x 1280 call, 1.9 TB/s)
__global__ void __launch_bounds__(256) k_layernorm8(const bf16_t* __restrict__ x, bf16_t* __restrict__ y, const bf16_t* __restrict__ w,
                                                    const bf16_t* __restrict__ bias, int d, float eps) {
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x, nch = d >> 3;
    const bool live = tid < nch;
    const int ch = live ? tid : 0;
    const uint4 xq = reinterpret_cast<const uint4*>(x + row * d)[ch];
    const uint4 wq = reinterpret_cast<const uint4*>(w)[ch];
    const uint4 bq = reinterpret_cast<const uint4*>(bias)[ch];
    const uint32_t xw[4] = {xq.x, xq.y, xq.z, xq.w}, ww[4] = {wq.x, wq.y, wq.z, wq.w}, bw[4] = {bq.x, bq.y, bq.z, bq.w};
    float v[8], s = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = bf16_to_f32((bf16_t)(xw[j] & 0xffffu)); v[2 * j + 1] = bf16_to_f32((bf16_t)(xw[j] >> 16));
        s += live ? v[2 * j] + v[2 * j + 1] : 0.0f;
    }
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)d;
    __syncthreads();
    float q = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float t = v[e] - mean; q += live ? t * t : 0.0f; }
    q = wave_sum(q);
    if ((tid & 63) == 0) red[tid >> 6] = q;
    __syncthreads();
    const float rstd = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)d + eps);
    if (live) {
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float w0 = bf16_to_f32((bf16_t)(ww[j] & 0xffffu)), w1 = bf16_to_f32((bf16_t)(ww[j] >> 16));
            const float b0 = bf16_to_f32((bf16_t)(bw[j] & 0xffffu)), b1 = bf16_to_f32((bf16_t)(bw[j] >> 16));
            o[j] = (uint32_t)f32_to_bf16((v[2 * j] - mean) * rstd * w0 + b0) | ((uint32_t)f32_to_bf16((v[2 * j + 1] - mean) * rstd * w1 + b1) << 16);
        }
        reinterpret_cast<uint4*>(y + row * d)[ch] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}
void launch_layernorm(const bf16_t* x, bf16_t* y, const bf16_t* w, const bf16_t* b, int rows, int d, float eps, hipStream_t s) {
    if (rows <= 0) return;
    const bool a16 = ((((uintptr_t)x) | ((uintptr_t)y) | ((uintptr_t)w) | ((uintptr_t)b)) & 15) == 0;
    if (d % 8 == 0 && d <= 2048 && a16) hipLaunchKernelGGL(k_layernorm8, dim3(rows), dim3(256), 0, s, x, y, w, b, d, eps);
    else hipLaunchKernelGGL(k_layernorm, dim3(rows), dim3(256), 0, s, x, y, w, b, d, eps);
}

// ============================================================================ conv stem patches
// out[(b*Tout + t)][k*C + c] = in[b][t*stride + k - 1][c]  (zero outside), k = 0..2   (Conv1d k3 p1, NLC)
template <typename TIN>
__global__ void k_im2col3(const TIN* __restrict__ in, bf16_t* __restrict__ out, int B, int Tin, int C, int Tout, int stride) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t total = (size_t)B * Tout * 3 * C;
    if (i >= total) return;
    int c = (int)(i % C);
    size_t r = i / C;
    int k = (int)(r % 3);
    r /= 3;
    int t = (int)(r % Tout);
    int b = (int)(r / Tout);
    int ti = t * stride + k - 1;
    float v = 0.0f;
    if (ti >= 0 && ti < Tin) {
        TIN raw = in[((size_t)b * Tin + ti) * C + c];
        if constexpr (sizeof(TIN) == 4) v = (float)raw; else v = bf16_to_f32((bf16_t)raw);
    }
    out[i] = f32_to_bf16(v);
}
void launch_im2col3_f32(const float* in, bf16_t* out, int B, int Tin, int C, int Tout, int stride, hipStream_t s) {
    size_t total = (size_t)B * Tout * 3 * C;
    hipLaunchKernelGGL((k_im2col3<float>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, in, out, B, Tin, C, Tout, stride);
}
void launch_im2col3_bf16(const bf16_t* in, bf16_t* out, int B, int Tin, int C, int Tout, int stride, hipStream_t s) {
    size_t total = (size_t)B * Tout * 3 * C;
    hipLaunchKernelGGL((k_im2col3<bf16_t>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, in, out, B, Tin, C, Tout, stride);
}

// ============================================================================ K / V -> tiled fragment caches
// src rows [B*T][ld]; K columns at kcol0 + h*D + d, V columns at vcol0 + h*D + d.
// kcache [B][H][Spad/32][2][D/32][64][8],  vcache [B][H][Spad/32][D/16][64][8]   (layouts of lm_kernels.hip)
// One block per (32-key tile, head, batch row): the tile's K and V rows (32 x D, read as 16-byte pieces of the source rows) go
// through LDS and leave as the tile's two contiguous 32*D*2-byte images, written with 16-byte stores - the element-wise version
// (2-byte stores, the V image strided by 16 B between neighbouring threads) moved 122 MB per large-v3 layer at 1.5 TB/s.
template <int D>
__global__ void __launch_bounds__(256) k_scatter_kv(const bf16_t* __restrict__ src, int ld, int kcol0, int vcol0, bf16_t* __restrict__ kc,
                                                    bf16_t* __restrict__ vc, int T, int H, int Spad) {
    __shared__ __attribute__((aligned(16))) bf16_t ks[32][D + 8];          // +8: rows 16 B apart in bank space
    __shared__ __attribute__((aligned(16))) bf16_t vs[32][D + 8];
    const int tile = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
    constexpr int CH = D / 8;                                                // 16-byte pieces per row
    for (int i = tid; i < 32 * CH; i += 256) {
        const int r = i / CH, c = i - r * CH;
        const int t = tile * 32 + r;
        uint4 kv = make_uint4(0, 0, 0, 0), vv = kv;
        if (t < T) {
            const bf16_t* row = src + ((size_t)b * T + t) * ld;
            kv = *reinterpret_cast<const uint4*>(row + kcol0 + h * D + c * 8);
            vv = *reinterpret_cast<const uint4*>(row + vcol0 + h * D + c * 8);
        }
        *reinterpret_cast<uint4*>(&ks[r][c * 8]) = kv;
        *reinterpret_cast<uint4*>(&vs[r][c * 8]) = vv;
    }
    __syncthreads();
    const size_t base = ((size_t)b * H + h) * (size_t)Spad * D + (size_t)tile * 32 * D;
    // K image [2][D/32][64][8]: lane = q*16 + prow holds key pr (prow = ((pr>>3)<<2)|(pr&3), half = (pr>>2)&1), dims dc*32 + q*8 .. +8
    for (int i = tid; i < 2 * (D / 32) * 64; i += 256) {
        const int lane = i & 63, dc = (i >> 6) % (D / 32), half = i / (64 * (D / 32));
        const int prow = lane & 15, q = lane >> 4;
        const int pr = ((prow >> 2) << 3) | (half << 2) | (prow & 3);
        *reinterpret_cast<uint4*>(kc + base + (size_t)i * 8) = *reinterpret_cast<const uint4*>(&ks[pr][dc * 32 + q * 8]);
    }
    // V image [D/16][64][8]: lane = (pr>>3)*16 + (d&15) holds keys (pr>>3)*8 .. +8 of dim dt*16 + (d&15)
    for (int i = tid; i < (D / 16) * 64; i += 256) {
        const int lane = i & 63, dt = i >> 6;
        const int d = dt * 16 + (lane & 15), p0 = (lane >> 4) * 8;
        bf16_t v8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v8[e] = vs[p0 + e][d];
        *reinterpret_cast<uint4*>(vc + base + (size_t)i * 8) = *reinterpret_cast<const uint4*>(v8);
    }
}
void launch_scatter_kv(const bf16_t* src, int ld, int kcol0, int vcol0, bf16_t* kc, bf16_t* vc, int B, int T, int H, int D,
                       int Spad, hipStream_t s) {
    MIS_REQUIRE((D == 64 || D == 128) && ld % 8 == 0 && kcol0 % 8 == 0 && vcol0 % 8 == 0 && Spad % 32 == 0, MIS_ERR_INVALID_INPUT,
                "K/V scatter: unsupported layout");
    dim3 grid(cdiv(T, 32), H, B);
    if (D == 64) hipLaunchKernelGGL((k_scatter_kv<64>), grid, dim3(256), 0, s, src, ld, kcol0, vcol0, kc, vc, T, H, Spad);
    else hipLaunchKernelGGL((k_scatter_kv<128>), grid, dim3(256), 0, s, src, ld, kcol0, vcol0, kc, vc, T, H, Spad);
}

// ============================================================================ encoder self attention (non causal)
//
// One 32-key tile of 16 queries: raw scores (lane = query j, key group g4: keys g4*8 + e) -> P as bf16 hi + lo in the P.V operand layout.  The softmax is
// bound by VALU issue (360 M scores per layer of 8 windows), so: p = 2^t, t = S c - m with c = scale log2 e in one fma; the maximum that p is
// taken against moves only when some t passes 8 (no cross-lane traffic on the usual tile; taken over t and not over S, a maximum needs no quieting of the matrix core's output) - the
// ratio numerator / denominator does not depend on it, and sums of at most 256 T stay far inside float32; hi / lo are converted two at a time.
struct AttnRow { float m = -INFINITY, l = 0.0f; };
template <bool MASKED>
__device__ __forceinline__ void attn_mask(f32x4_t& S0, f32x4_t& S1, int key0, int T) {
    if constexpr (MASKED) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float& s = e < 4 ? reinterpret_cast<float*>(&S0)[e] : reinterpret_cast<float*>(&S1)[e - 4];
            s = key0 + e < T ? s : -INFINITY;
        }
    }
}
__device__ __forceinline__ float attn_shift(const f32x4_t& S0, const f32x4_t& S1, float c, const AttnRow& r, float (&t)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = fmaf(e < 4 ? S0[e] : S1[e - 4], c, -r.m);
    return fmaxf(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])), fmaxf(fmaxf(t[4], t[5]), fmaxf(t[6], t[7])));
}
// the maximum moves (all of the wave's rows): the output so far and the sum are scaled
template <int ND>
__device__ __forceinline__ void attn_move(const f32x4_t& S0, const f32x4_t& S1, float c, AttnRow& r, float (&t)[8], f32x4_t (&O)[ND], int g4) {
    float mx = fmaxf(fmaxf(fmaxf(S0[0], S0[1]), fmaxf(S0[2], S0[3])), fmaxf(fmaxf(S1[0], S1[1]), fmaxf(S1[2], S1[3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(r.m, mx * c), alpha = __builtin_amdgcn_exp2f(r.m - m_new);       // (first tile: 2^-inf = 0)
    r.m = m_new;
    r.l *= alpha;
    float ar[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) ar[q] = __shfl(alpha, g4 * 4 + q, 64);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q) O[dt][q] *= ar[q];
    (void)attn_shift(S0, S1, c, r, t);
}
__device__ __forceinline__ void attn_probs(const float (&t)[8], AttnRow& r, bf16x8_t& ph, bf16x8_t& pl) {
    typedef float f2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 h2_t __attribute__((ext_vector_type(2)));
    float psum = 0.0f;
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(t[e]), p1 = __builtin_amdgcn_exp2f(t[e + 1]);
        psum = e ? psum + p0 : p0;
        psum += p1;
        const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){p0, p1}, h2_t));
        hw[e >> 1] = h;
        lw[e >> 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){p0 - __uint_as_float(h << 16), p1 - __uint_as_float(h & 0xffff0000u)}, h2_t));
    }
    r.l += psum;
    ph = __builtin_bit_cast(bf16x8_t, make_uint4(hw[0], hw[1], hw[2], hw[3]));
    pl = __builtin_bit_cast(bf16x8_t, make_uint4(lw[0], lw[1], lw[2], lw[3]));
}
// grid (ceil(T/64), H, B), 4 waves x 16 query rows.  S^T = K Q^T (A = K fragment, B = Q^T): lane (q row j, group g4)
// holds the scores of keys base + g4*8 + e; online softmax per query row; O += P V with P split into bf16 hi + lo.
template <int D>
__global__ void __launch_bounds__(256) k_attn_prefill(const bf16_t* __restrict__ q, int ldq, const bf16_t* __restrict__ kc,
                                                      const bf16_t* __restrict__ vc, bf16_t* __restrict__ out, int ldo,
                                                      int T, int H, int Spad, float scale) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int b = blockIdx.z, h = blockIdx.y, t0 = blockIdx.x * 64 + wave * 16;
    if (t0 >= T) return;
    const int j = lane & 15, g4 = lane >> 4;
    const int tq = t0 + j;
    bf16x8_t qf[D / 32];
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
        if (tq < T) qf[c] = *reinterpret_cast<const bf16x8_t*>(q + ((size_t)b * T + tq) * ldq + h * D + c * 32 + g4 * 8);
        else qf[c] = (bf16x8_t){0, 0, 0, 0, 0, 0, 0, 0};
    }
    const size_t base = ((size_t)b * H + h) * (size_t)Spad * D;
    const bf16x8_t* kbase = reinterpret_cast<const bf16x8_t*>(kc + base) + lane;
    const bf16x8_t* vbase = reinterpret_cast<const bf16x8_t*>(vc + base) + lane;
    f32x4_t O[D / 16];
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) O[dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    AttnRow row;
    const float sc2 = scale * 1.4426950408889634f;
    const int n_tiles = (T + 31) >> 5;
    for (int tile = 0; tile < n_tiles; ++tile) {
        const int kb = tile * 32;
        f32x4_t S0 = (f32x4_t){0.f, 0.f, 0.f, 0.f}, S1 = S0;
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
            bf16x8_t a0 = kbase[((size_t)tile * 2) * (D / 32) * 64 + c * 64];
            bf16x8_t a1 = kbase[((size_t)tile * 2 + 1) * (D / 32) * 64 + c * 64];
            S0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, qf[c], S0, 0, 0, 0);
            S1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, qf[c], S1, 0, 0, 0);
        }
        bf16x8_t ph, pl;
        float t[8];
        attn_mask<true>(S0, S1, kb + g4 * 8, T);
        if (__any(attn_shift(S0, S1, sc2, row, t) > 8.0f)) attn_move(S0, S1, sc2, row, t, O, g4);
        attn_probs(t, row, ph, pl);
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            bf16x8_t vb = vbase[((size_t)tile * (D / 16) + dt) * 64];
            f32x4_t o = O[dt];
            o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vb, o, 0, 0, 0);
            o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vb, o, 0, 0, 0);
            O[dt] = o;
        }
    }
    float l_run = row.l;
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    // O[dt][r]: row = query (g4*4 + r), col = d (dt*16 + j); the row's normaliser lives in lane (g4*4 + r)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float lr = __shfl(l_run, g4 * 4 + r, 64);
        int tr = t0 + g4 * 4 + r;
        if (tr < T) {
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt)
                out[((size_t)b * T + tr) * ldo + h * D + dt * 16 + j] = f32_to_bf16(O[dt][r] / lr);
        }
    }
}
// ---- the same attention on 256-row blocks.  What the kernel above costs per 32-key tile and wave: 16 fragment loads straight from global memory, waited
// for where they are used, for 12 MFMAs on 16 query rows - and every one of the 94 waves of a head streams the head's whole 393 KB of K/V for itself.
// Here a block is 256 query rows (8 waves x 2 groups of 16): the tile's K and V images (8 KB, already in fragment order - lm_kernels.hip's cache
// tiling) are staged ONCE per block through LDS, one 16-byte piece per thread, tile t + 1 requested before tile t is multiplied (two LDS buffers, one
// barrier per tile); a wave reads each fragment once (lane-linear ds_read_b128, conflict-free) and uses it for both of its row groups: 24 MFMAs per 8 LDS
// reads.  The key mask is applied on the last tile only.  Same operations per query row in the same order as k_attn_prefill: results are bit-identical
// (tests/test_gpu_whisper.py).  Bound: the softmax's VALU work (issued in 71 % of the cycles; MFMA 41 %): 149 - 158 us per layer of 8 windows x 20 heads.  228 with the
// maximum taken over the raw scores, the row groups one after the other and the mask inside the loop; 260 with the score's scale, its logarithm base and a cross-lane maximum per
// tile there as well; that form with two tiles per barrier 251.
template <int D>
__global__ void __launch_bounds__(512, 4) k_attn_prefill2(const bf16_t* __restrict__ q, int ldq, const bf16_t* __restrict__ kc,
                                                          const bf16_t* __restrict__ vc, bf16_t* __restrict__ out, int ldo,
                                                          int T, int H, int Spad, float scale) {
    static_assert(D == 64, "one 16-byte piece of the tile's 8 KB per thread");
    constexpr int NW = 8, QR = 32 * NW, IMG = 32 * D;                // bf16 elements of one K (or V) tile image
    __shared__ __attribute__((aligned(16))) bf16_t kv[2][2 * IMG];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b = blockIdx.z, h = blockIdx.y, q0 = blockIdx.x * QR + wave * 32;
    const int j = lane & 15, g4 = lane >> 4;
    bf16x8_t qf[2][D / 32];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int tq = q0 + 16 * g + j;
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
            if (tq < T) qf[g][c] = *reinterpret_cast<const bf16x8_t*>(q + ((size_t)b * T + tq) * ldq + h * D + c * 32 + g4 * 8);
            else qf[g][c] = (bf16x8_t){0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    const size_t base = ((size_t)b * H + h) * (size_t)Spad * D;
    // staging: threads 0 .. 255 move the K image, 256 .. 511 the V image (IMG / 8 = 256 pieces each)
    const uint4* src = reinterpret_cast<const uint4*>((tid < 256 ? kc : vc) + base) + (tid & 255);
    const int dst_piece = tid;                                            // K image first, V image behind it
    const int n_tiles = (T + 31) >> 5;
    uint4 st = src[0];
    *(reinterpret_cast<uint4*>(kv[0]) + dst_piece) = st;
    __syncthreads();
    f32x4_t O[2][D / 16];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) O[g][dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    AttnRow row[2];
    const float sc2 = scale * 1.4426950408889634f;
    auto tile_math = [&](int tile, const bf16_t* img, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        const int kb = tile * 32;
        const bf16x8_t* kf = reinterpret_cast<const bf16x8_t*>(img) + lane;
        const bf16x8_t* vf = reinterpret_cast<const bf16x8_t*>(img + IMG) + lane;
        bf16x8_t a0[D / 32], a1[D / 32], vb[D / 16];
#pragma unroll
        for (int c = 0; c < D / 32; ++c) { a0[c] = kf[c * 64]; a1[c] = kf[((D / 32) + c) * 64]; }
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) vb[dt] = vf[dt * 64];
        f32x4_t S0[2], S1[2];
        float t[2][8], mx[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            S0[g] = S1[g] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < D / 32; ++c) {
                S0[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[c], qf[g][c], S0[g], 0, 0, 0);
                S1[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[c], qf[g][c], S1[g], 0, 0, 0);
            }
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            attn_mask<MASKED>(S0[g], S1[g], kb + g4 * 8, T);
            mx[g] = attn_shift(S0[g], S1[g], sc2, row[g], t[g]);
        }
        if (__any(fmaxf(mx[0], mx[1]) > 8.0f)) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
                if (__any(mx[g] > 8.0f)) attn_move(S0[g], S1[g], sc2, row[g], t[g], O[g], g4);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            bf16x8_t ph, pl;
            attn_probs(t[g], row[g], ph, pl);
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) {
                f32x4_t o = O[g][dt];
                o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vb[dt], o, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vb[dt], o, 0, 0, 0);
                O[g][dt] = o;
            }
        }
    };
    // (the last tile on its own: with its mask inside the loop the outputs are copied between the two forms' registers, 38 moves a tile)
    for (int tile = 0; tile + 1 < n_tiles; ++tile) {
        st = src[(size_t)(tile + 1) * (IMG / 8)];
        tile_math(tile, kv[tile & 1], std::false_type{});
        *(reinterpret_cast<uint4*>(kv[(tile + 1) & 1]) + dst_piece) = st;
        __syncthreads();
    }
    tile_math(n_tiles - 1, kv[(n_tiles - 1) & 1], std::true_type{});
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        float lr_all = row[g].l;
        lr_all += __shfl_xor(lr_all, 16, 64);
        lr_all += __shfl_xor(lr_all, 32, 64);
        // O[g][dt][r]: row = query (g4*4 + r), col = d (dt*16 + j); the row's normaliser lives in lane (g4*4 + r)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float lr = __shfl(lr_all, g4 * 4 + r, 64);
            const int tr = q0 + 16 * g + g4 * 4 + r;
            if (tr < T) {
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt)
                    out[((size_t)b * T + tr) * ldo + h * D + dt * 16 + j] = f32_to_bf16(O[g][dt][r] / lr);
            }
        }
    }
}
void launch_attn_prefill(const bf16_t* q, int ldq, const bf16_t* kc, const bf16_t* vc, bf16_t* out, int ldo, int B, int T,
                         int H, int D, int Spad, hipStream_t s) {
    float scale = 1.0f / sqrtf((float)D);
    const char* ve = getenv("MIS_ATTN_PREFILL_V1");                      // tests: the 16-rows-per-wave kernel (read per launch)
    const bool v1 = ve && atoi(ve) != 0;
    if (D == 64 && !v1 && ((uintptr_t)kc & 15) == 0 && ((uintptr_t)vc & 15) == 0) {
        hipLaunchKernelGGL((k_attn_prefill2<64>), dim3(cdiv(T, 256), H, B), dim3(512), 0, s, q, ldq, kc, vc, out, ldo, T, H, Spad, scale);
        return;
    }
    dim3 grid(cdiv(T, 64), H, B), block(256);
    if (D == 64) hipLaunchKernelGGL((k_attn_prefill<64>), grid, block, 0, s, q, ldq, kc, vc, out, ldo, T, H, Spad, scale);
    else if (D == 128) hipLaunchKernelGGL((k_attn_prefill<128>), grid, block, 0, s, q, ldq, kc, vc, out, ldo, T, H, Spad, scale);
    else throw MisError(MIS_ERR_INVALID_INPUT, "head_dim must be 64 or 128");
}

// ============================================================================ decoder step helpers
// h = T(E[tok] + P[pos]) ; x = LayerNorm(h) packed ; advances positions like k_embed_rmsnorm
__global__ void __launch_bounds__(256) k_whisper_embed_ln(const bf16_t* __restrict__ emb, const bf16_t* __restrict__ pos_emb,
                                                          const int32_t* __restrict__ ids, const uint8_t* __restrict__ active,
                                                          int* __restrict__ pos_cur, int* __restrict__ pos_next,
                                                          const bf16_t* __restrict__ lw, const bf16_t* __restrict__ lb,
                                                          bf16_t* __restrict__ h, bf16_t* __restrict__ x, int d, int vocab,
                                                          int max_pos, int batch) {
    __shared__ float red[4];
    const int m = blockIdx.x, MT = gridDim.x >> 4;
    int id = (m < batch) ? ids[m] : 0;
    if (id < 0 || id >= vocab) id = 0;
    int p = (m < batch) ? pos_next[m] : 0;
    if (threadIdx.x == 0 && m < batch) {
        pos_cur[m] = p;
        if (active[m]) pos_next[m] = p + 1;
    }
    if (p >= max_pos) p = max_pos - 1;
    float s = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) {
        float v = bf16_round_f32(bf16_to_f32(emb[(size_t)id * d + i]) + bf16_to_f32(pos_emb[(size_t)p * d + i]));
        h[(size_t)m * d + i] = f32_to_bf16(v);
        s += v;
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)d;
    __syncthreads();
    float q = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) { float t = bf16_to_f32(h[(size_t)m * d + i]) - mean; q += t * t; }
    q = wave_sum(q);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
    __syncthreads();
    const float rstd = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)d + 1e-5f);
    for (int i = threadIdx.x; i < d; i += 256) {
        float f = bf16_to_f32(h[(size_t)m * d + i]);
        size_t off = ((((size_t)(i >> 5) * MT + (m >> 4)) * 64) + (((i & 31) >> 3) << 4) + (m & 15)) * 8 + (i & 7);
        x[off] = f32_to_bf16((f - mean) * rstd * bf16_to_f32(lw[i]) + bf16_to_f32(lb[i]));
    }
}
void launch_whisper_embed_ln(const bf16_t* emb, const bf16_t* pos_emb, const int32_t* ids, const uint8_t* active, int* pos_cur,
                             int* pos_next, const bf16_t* lw, const bf16_t* lb, bf16_t* h, bf16_t* x, int d, int vocab,
                             int max_pos, int batch, int Mpad, hipStream_t s) {
    hipLaunchKernelGGL(k_whisper_embed_ln, dim3(Mpad), dim3(256), 0, s, emb, pos_emb, ids, active, pos_cur, pos_next, lw, lb, h,
                       x, d, vocab, max_pos, batch);
}

// suppress masks of the greedy loop (WhisperModel.swift:228-236,293-309): logits += -1e9 on the listed ids
// (begin list only while the row has generated nothing); ids >= timestamp_begin are excluded via the sampler range.
__global__ void k_whisper_suppress(bf16_t* __restrict__ logits, int Vpad, int vocab, const int32_t* __restrict__ sup, int n_sup,
                                   const int32_t* __restrict__ bsup, int n_bsup, const int32_t* __restrict__ n_gen,
                                   const uint8_t* __restrict__ active) {
    const int b = blockIdx.x;
    if (active && !active[b]) return;
    bf16_t* l = logits + (size_t)b * Vpad;
    for (int i = threadIdx.x; i < n_sup; i += blockDim.x) {
        int id = sup[i];
        if (id >= 0 && id < vocab) l[id] = f32_to_bf16(bf16_to_f32(l[id]) + -1e9f);
    }
    if (n_gen[b] == 0)
        for (int i = threadIdx.x; i < n_bsup; i += blockDim.x) {
            int id = bsup[i];
            bool dup = false;
            for (int k = 0; k < n_sup; ++k) dup = dup || (sup[k] == id);
            if (id >= 0 && id < vocab && !dup) l[id] = f32_to_bf16(bf16_to_f32(l[id]) + -1e9f);
        }
}
void launch_whisper_suppress(bf16_t* logits, int Vpad, int vocab, const int32_t* sup, int n_sup, const int32_t* bsup, int n_bsup,
                             const int32_t* n_gen, const uint8_t* active, int batch, hipStream_t s) {
    if (n_sup + n_bsup == 0) return;
    hipLaunchKernelGGL(k_whisper_suppress, dim3(batch), dim3(128), 0, s, logits, Vpad, vocab, sup, n_sup, bsup, n_bsup, n_gen, active);
}
