// lm_prefill.hip - the prompt as ONE [positions x rows] pass: compute-bound MFMA GEMMs over the packed LM weights.
//
// Reference being replaced: the prefill call of the generate loop, `model(inputIds [1, L], cache:)` (LlamaTTS.swift:711), which runs
// the whole prompt through every layer at once.  The decode engine used to feed the prompt one position per step (L weight-streaming
// passes: 56 ms of the 1.6 s bench job for 32-token prompts, and linear in L - voice-cloning prompts carry hundreds of audio tokens).
// Here all L x B prompt tokens form the M dimension of four GEMMs per layer (M = 1024 at the bench shape), each weight byte is read
// once per CHUNK of positions instead of once per position, and the attention takes the chunk's queries together over the decode step's
// caches.  Rows are PACKED: the chunk's positions of sequence 0, then those of sequence 1, ... - no row stands for the padding of a shorter prompt
// (prompts of 300 .. 450 tokens padded to 450: 15 % of every GEMM).
//
//   k_pf_embed_rmsnorm  h[r] = E[token(b, t)], x[r] = RMSNorm(h[r]) (row-major); active / position tables for the short-prompt form
//   k_gemm_pf<EPI>      C[M][N] = X[M][K] . W^T with W in the decode path's packed MFMA-A tile layout [N/16][K/32][64][8]:
//                       a weight fragment is one 1 KiB global_load_lds piece and its LDS image IS the A fragment (lane-linear:
//                       ds_read_b128 at lane*16, conflict free); X tiles as in k_gemm_big2 (whisper_kernels.hip: source-side
//                       XOR swizzle).  128 x 128 x 64 tiles, two LDS buffers, one barrier per k-step.  Epilogues:
//                         PF_ROWS_BF16  T(acc) [M][N]                    (q|k|v)
//                         PF_RESID  h = T(h + T(acc)) in place, bf16      (o_proj, down_proj: LlamaTTS.swift:306-309)
//                         PF_SILU   act = T(T(g T(sigmoid g)) u), gate / up tiles interleaved as packed (:283)
//   k_gemm_pf_wide      the same on tiles of 128 .. 192 x 256, four waves (gemm_tiles.h): many rows
//   k_gemm_pf_ring      the same on tiles of 32 x 32: few rows
//   k_gemm_pf_codes     the same on 8- and 4-bit codes, more than 64 rows (fewer, and up to 96 of large 4-bit matrices: k_gemm_skinny_q, lm_qgemm.hip, the same bits)
//   k_pf_rope_append    q|k|v of the chunk -> roped queries (bf16 rows) and the tiled K / V caches of the decode step
//   k_pf_attn           causal attention of the chunk's queries over the caches (MFMA, K / V tiles shared by 128 or 256 queries)
//   k_pf_rmsnorm        x[r] = RMSNorm(h[r]) row-major
//   k_pf_pack_last      every sequence's last row -> the packed x operand of the decode step (lm_head of the first new token)
//   k_pf_pack_rows      rows -> packed x operand of a slice of k_gemm_skinny_q
// Rounding points are those of the decode step (bf16 at every MLX primitive boundary); only float32 summation orders differ.
#include "common.h"
#include "gemm_tiles.h"
#include "lm_kernels.h"

#include <type_traits>

#define PF_BM 128
#define PF_BN 128
#define PF_BK 64

__device__ __forceinline__ float pf_block_sum_256(float v, float* red) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    const float t = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return t;
}

// The chunk [t0, t0 + tc) of left-padded prompts: sequence b has n = hi - lo positions [lo, hi) in it, position p is packed row row0 + p
struct PfSpan { int lo, hi, row0; };
__device__ __forceinline__ int pf_count(const int32_t* lens, int b, int Lmax, int t0, int tc, int& lo) {
    const int shift = Lmax - lens[b] - t0;
    lo = max(0, -shift);
    return max(0, tc - shift - lo);
}
__device__ __forceinline__ PfSpan pf_span(const int32_t* lens, int b, int Lmax, int t0, int tc) {
    int row = 0, lo;
    for (int i = 0; i < b; ++i) row += pf_count(lens, i, Lmax, t0, tc, lo);
    const int n = pf_count(lens, b, Lmax, t0, tc, lo);
    return PfSpan{lo, lo + n, row - lo};
}
// (sequence, left-padded position) of row r; Mpad = 0: packed rows, else row t * Mpad + b
__device__ __forceinline__ bool pf_row(const int32_t* lens, int r, int Lmax, int t0, int tc, int batch, int Mpad, int& b, int& t) {
    if (Mpad) {
        const int tl = r / Mpad;
        b = r - tl * Mpad; t = t0 + tl;
        return b < batch && t >= Lmax - lens[b];
    }
    for (b = 0; b < batch; ++b) {
        int lo;
        const int n = pf_count(lens, b, Lmax, t0, tc, lo);
        if (r < n) { t = Lmax - lens[b] + lo + r; return true; }
        r -= n;
    }
    b = 0; t = t0;
    return false;
}
// one 256-thread block per row of the chunk [t0, t0 + tc)
__global__ void __launch_bounds__(256) k_pf_embed_rmsnorm(const bf16_t* __restrict__ emb, const int32_t* __restrict__ prompt /*[batch][Lmax] left padded*/,
                                                          const int32_t* __restrict__ lens, int Lmax, int t0, int tc, int batch, int Mpad, int vocab,
                                                          const bf16_t* __restrict__ wnorm, bf16_t* __restrict__ h, bf16_t* __restrict__ x,
                                                          int32_t* __restrict__ pos_tab, uint8_t* __restrict__ act_tab, int d, float eps) {
    __shared__ float red[4];
    const int r = blockIdx.x;
    int b, t;
    const bool on = pf_row(lens, r, Lmax, t0, tc, batch, Mpad, b, t);
    if (pos_tab && threadIdx.x == 0) { pos_tab[r] = on ? t - (Lmax - lens[b]) : 0; act_tab[r] = on ? 1 : 0; }
    int id = on ? prompt[(size_t)b * Lmax + t] : -1;
    if (id >= vocab) id = -1;
    const bf16_t* e = emb + (size_t)(id < 0 ? 0 : id) * d;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) {
        const bf16_t v = id < 0 ? (bf16_t)0 : e[i];
        h[(size_t)r * d + i] = v;
        const float f = bf16_to_f32(v);
        ss += f * f;
    }
    const float inv = 1.0f / sqrtf(pf_block_sum_256(ss, red) / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256) {
        const float f = id < 0 ? 0.0f : bf16_to_f32(e[i]);
        x[(size_t)r * d + i] = f32_to_bf16(bf16_to_f32(wnorm[i]) * bf16_round_f32(f * inv));       // T(w * T(x * rsqrt(mean + eps)))
    }
}
// the same for engines that feed input embeddings instead of token ids (Qwen3-TTS talker): rows [Lmax][src_rows][d] computed by the
// caller; `Mpad` here and in k_pf_embed_rmsnorm is the chunk's rows per position (the batch), 0 for packed rows
__global__ void __launch_bounds__(256) k_pf_rows_rmsnorm(const bf16_t* __restrict__ rows, int src_rows, const int32_t* __restrict__ lens, int Lmax, int t0, int tc, int batch,
                                                         int Mpad, const bf16_t* __restrict__ wnorm, bf16_t* __restrict__ h, bf16_t* __restrict__ x,
                                                         int32_t* __restrict__ pos_tab, uint8_t* __restrict__ act_tab, int d, float eps) {
    __shared__ float red[4];
    const int r = blockIdx.x;
    int b, t;
    const bool on = pf_row(lens, r, Lmax, t0, tc, batch, Mpad, b, t);
    if (pos_tab && threadIdx.x == 0) { pos_tab[r] = on ? t - (Lmax - lens[b]) : 0; act_tab[r] = on ? 1 : 0; }
    const bf16_t* e = rows + ((size_t)t * src_rows + b) * d;                   // the caller's matrix keeps its own rows per position
    float ss = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) {
        const bf16_t v = on ? e[i] : (bf16_t)0;
        h[(size_t)r * d + i] = v;
        const float f = bf16_to_f32(v);
        ss += f * f;
    }
    const float inv = 1.0f / sqrtf(pf_block_sum_256(ss, red) / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256) {
        const float f = on ? bf16_to_f32(e[i]) : 0.0f;
        x[(size_t)r * d + i] = f32_to_bf16(bf16_to_f32(wnorm[i]) * bf16_round_f32(f * inv));
    }
}
__global__ void __launch_bounds__(256) k_pf_rmsnorm(const bf16_t* __restrict__ h, const bf16_t* __restrict__ wnorm, bf16_t* __restrict__ x,
                                                    int d, float eps) {
    __shared__ float red[4];
    const size_t r = blockIdx.x;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < d; i += 256) { const float f = bf16_to_f32(h[r * d + i]); ss += f * f; }
    const float inv = 1.0f / sqrtf(pf_block_sum_256(ss, red) / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256)
        x[r * d + i] = f32_to_bf16(bf16_to_f32(wnorm[i]) * bf16_round_f32(bf16_to_f32(h[r * d + i]) * inv));
}
// the row of every sequence's last position (packed rows; Mpad - batch rows of zeros behind them) -> packed MFMA-B fragments of the decode step's x operand
__global__ void k_pf_pack_last(const bf16_t* __restrict__ rows, const int32_t* __restrict__ lens, int Lmax, int t0, int tc, int batch, bf16_t* __restrict__ xpk, int d, int MT) {
    const int m = blockIdx.x;
    const PfSpan sp = pf_span(lens, min(m, batch - 1), Lmax, t0, tc);
    const bool on = m < batch && sp.hi > sp.lo;                    // (an empty prompt has no row)
    const bf16_t* src = rows + (size_t)(on ? sp.row0 + sp.hi - 1 : 0) * d;
    for (int k = threadIdx.x; k < d; k += blockDim.x) xpk[xpk_index(m, k, MT)] = on ? src[k] : (bf16_t)0;
}
// rows [Mpad][d] row-major -> packed MFMA-B fragments of the decode step's x operand
__global__ void k_pf_pack_rows(const bf16_t* __restrict__ rows, bf16_t* __restrict__ xpk, int d, int MT) {
    const int m = blockIdx.x;
    for (int k = threadIdx.x; k < d; k += blockDim.x) xpk[xpk_index(m, k, MT)] = rows[(size_t)m * d + k];
}

struct PfGemmParams {
    const bf16_t* X;      // [M][K] row-major
    const bf16_t* Wp;     // packed [NT][KT][64][8]
    void* C;              // PF_F32: float [M][N]; PF_RESID: bf16 h [M][N] (read-modify-write); PF_SILU: bf16 act [M][N/2]
    int M, N, K;          // N = rows of W (PF_SILU: 2 * ff, gate / up tiles interleaved)
    PfExtra ex;           // the epilogues of layer-list models (lm_blocks.hip)
};

// epilogue of TN x TM MFMA tiles, the first at W rows 16 tile0 and X rows m0
template <int EPI, int TN, int TM>
__device__ __forceinline__ void pf_epilogue(const PfGemmParams& p, const f32x4_t (&acc)[TN][TM], int tile0, int m0, int lane) {
    // epilogue.  C/D lane l, reg e: W row (n) = 16*tile + (l >> 4)*4 + e, X row (m) = l & 15
    const int nl = (lane >> 4) * 4, NT = p.N >> 4;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = m0 + j * 16 + (lane & 15);
        if (m >= p.M) continue;
        if (EPI == PF_SILU || EPI == PF_SWIGLU) {
            bf16_t* act = reinterpret_cast<bf16_t*>(p.C);
            const int ff = p.N >> 1;
#pragma unroll
            for (int i = 0; i + 1 < TN; i += 2) {             // tile pair (gate, up) -> feature tile
                const int tile = tile0 + i;
                if (tile + 1 >= NT) continue;             // (tile, tile + 1) = (gate, up) of feature tile `tile >> 1`
                uint16_t res[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (EPI == PF_SWIGLU) {
                        const float gf = acc[i][j][e];
                        res[e] = f32_to_bf16(gf / (1.0f + __expf(-gf)) * acc[i + 1][j][e]);
                        continue;
                    }
                    const float g = bf16_round_f32(acc[i][j][e]);
                    const float u = bf16_round_f32(acc[i + 1][j][e]);
                    const float sg = bf16_round_f32(1.0f / (1.0f + __expf(-g)));
                    const float av = bf16_round_f32(g * sg);
                    res[e] = f32_to_bf16(av * u);
                }
                uint2 v;
                v.x = (uint32_t)res[0] | ((uint32_t)res[1] << 16);
                v.y = (uint32_t)res[2] | ((uint32_t)res[3] << 16);
                *reinterpret_cast<uint2*>(act + (size_t)m * ff + (tile >> 1) * 16 + nl) = v;
            }
        } else {
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int tile = tile0 + i;
                if (tile >= NT) continue;
                const int n = tile * 16 + nl;
                if constexpr (EPI >= PF_SPLIT_RELU2 && EPI != PF_SWIGLU) {
                    float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                    float* c32 = reinterpret_cast<float*>(p.C) + (size_t)m * p.ex.ldc + n;
                    if (EPI == PF_ACT_ROWS) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float sg = 1.0f / (1.0f + __expf(-v[e]));
                            v[e] = tile < p.ex.split ? v[e] * sg : sg;
                        }
                        *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.C) + (size_t)m * p.ex.ldc + n) =
                            make_uint2((uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16), (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16));
                    } else if (EPI == PF_ROWS_BF16 || (EPI == PF_SPLIT_RELU2 && tile >= p.ex.split)) {
                        uint16_t res[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (EPI == PF_SPLIT_RELU2) { const float t = fmaxf(v[e], 0.0f); v[e] = t * t; }
                            res[e] = f32_to_bf16(v[e]);
                        }
                        bf16_t* o = EPI == PF_ROWS_BF16 ? reinterpret_cast<bf16_t*>(p.C) + (size_t)m * p.ex.ldc + n
                                                        : reinterpret_cast<bf16_t*>(p.ex.out2) + (size_t)m * p.ex.ld2 + (n - p.ex.split * 16);
                        *reinterpret_cast<uint2*>(o) = make_uint2((uint32_t)res[0] | ((uint32_t)res[1] << 16), (uint32_t)res[2] | ((uint32_t)res[3] << 16));
                    } else if (EPI == PF_SCALED_ADD) {
                        const uint2 lw = *reinterpret_cast<const uint2*>(p.ex.ls + n);
                        const float l[4] = {bf16_to_f32((bf16_t)(lw.x & 0xffffu)), bf16_to_f32((bf16_t)(lw.x >> 16)), bf16_to_f32((bf16_t)(lw.y & 0xffffu)),
                                            bf16_to_f32((bf16_t)(lw.y >> 16))};
                        const float4 o = *reinterpret_cast<const float4*>(c32);
                        *reinterpret_cast<float4*>(c32) = make_float4(o.x + l[0] * v[0], o.y + l[1] * v[1], o.z + l[2] * v[2], o.w + l[3] * v[3]);
                    } else {
                        if (EPI == PF_SOFTCAP) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) { const float t = v[e] * p.ex.scale; v[e] = p.ex.cap > 0.0f ? p.ex.cap * tanhf(t / p.ex.cap) : t; }
                        }
                        *reinterpret_cast<float4*>(c32) = make_float4(v[0], v[1], v[2], v[3]);
                    }
                } else if (EPI == PF_F32) {
                    *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.C) + (size_t)m * p.N + n) =
                        make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
                } else {
                    bf16_t* h = reinterpret_cast<bf16_t*>(p.C) + (size_t)m * p.N + n;
                    const uint2 old = *reinterpret_cast<const uint2*>(h);
                    const uint32_t ow[2] = {old.x, old.y};
                    uint16_t res[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float hv = bf16_to_f32((bf16_t)((ow[e >> 1] >> (16 * (e & 1))) & 0xffffu));
                        res[e] = f32_to_bf16(hv + bf16_round_f32(acc[i][j][e]));                  // h = T(h + T(x W^T))
                    }
                    uint2 v;
                    v.x = (uint32_t)res[0] | ((uint32_t)res[1] << 16);
                    v.y = (uint32_t)res[2] | ((uint32_t)res[3] << 16);
                    *reinterpret_cast<uint2*>(h) = v;
                }
            }
        }
    }
}

template <int EPI>
__global__ void __launch_bounds__(256, 2) k_gemm_pf(PfGemmParams p) {
    __shared__ __attribute__((aligned(1024))) bf16_t Ws[2][PF_BN * PF_BK];
    __shared__ __attribute__((aligned(1024))) bf16_t Xs[2][PF_BM * PF_BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * PF_BN, m0 = blockIdx.y * PF_BM;
    if (n0 >= p.N) return;                              // (padding of the grid, see launch_gemm_pf)
    const int wn = wave >> 1, wm = wave & 1;            // wave tile: 64 n x 64 m
    const int NT = p.N >> 4, KT = p.K >> 5;
    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // staging.  W: fragment f = wave*4 + q of the 8 n-tiles x 2 k-tiles of a k-step, 1 KiB each, lane-linear both in memory and in LDS.
    // X: piece q of wave w = rows (w*4 + q)*8 .. +8, lane l -> row + (l >> 3), 16-byte position l & 7 holding chunk (l & 7) ^ ((row >> 1) & 7)
    const bf16_t* wsrc[4];
    const bf16_t* xsrc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int f = wave * 4 + q, ntl = f >> 1, ktl = f & 1;
        const int nt = min((n0 >> 4) + ntl, NT - 1);
        wsrc[q] = p.Wp + ((size_t)nt * KT + ktl) * 512 + lane * 8;
        const int r = (wave * 4 + q) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        const int xm = min(m0 + r, p.M - 1);
        if constexpr (EPI == PF_ROWS_BF16) xsrc[q] = p.X + (size_t)(p.ex.xrow ? p.ex.xrow[xm] : xm) * p.ex.ldx + chunk * 8;
        else xsrc[q] = p.X + (size_t)xm * p.K + chunk * 8;
    }
    auto stage = [&](int buf, int ks) {                  // k-step ks covers k-tiles 2 ks, 2 ks + 1 = columns 64 ks .. +64
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int f = wave * 4 + q;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wsrc[q] + (size_t)ks * 1024),
                                             (__attribute__((address_space(3))) void*)&Ws[buf][f * 512], 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xsrc[q] + ks * PF_BK),
                                             (__attribute__((address_space(3))) void*)&Xs[buf][(wave * 4 + q) * 8 * PF_BK], 16, 0, 0);
        }
    };
    const int sw = (lane >> 1) & 7;
    const int KS = p.K / PF_BK;
    stage(0, 0);
    for (int ks = 0; ks < KS; ++ks) {
        __syncthreads();                                 // this wave's LDS-DMA has landed (vmcnt(0)), then everybody's: k-step ks complete
        const bf16_t* wt = Ws[ks & 1];
        const bf16_t* xt = Xs[ks & 1];
        bf16x8_t a[2][4], b[2][4];                       // all fragment reads first, then the next DMA (see k_gemm_big2)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int pos = ((kk * 4 + (lane >> 4)) ^ sw) * 8;
#pragma unroll
            for (int i = 0; i < 4; ++i) a[kk][i] = *reinterpret_cast<const bf16x8_t*>(wt + ((wn * 4 + i) * 2 + kk) * 512 + lane * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[kk][j] = *reinterpret_cast<const bf16x8_t*>(xt + (wm * 64 + j * 16 + (lane & 15)) * PF_BK + pos);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ks + 1 < KS) stage((ks + 1) & 1, ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][i], b[kk][j], acc[i][j], 0, 0, 0);
    }
    pf_epilogue<EPI, 4, 4>(p, acc, (n0 >> 4) + wn * 4, m0 + wm * 64, lane);
}

// Many rows: tiles of 32 TM rows x 256 columns on four waves (gemm_tiles.h), persistent blocks.  Orpheus-3B, 3600 rows, us per launch, k_gemm_pf / here: gate | up
// 348 / 318, q|k|v 134 / 115, o and down together 160 / 121 on average (696 tiles of 128 x 128 are 1.4 rounds of 512 blocks; 228 tiles of 192 rows one
// of 256).  TM: the rounds decide - o and down at 3075 rows: 240 tiles with TM 5 132 us, 204 with TM 6 148, 300 with
// TM 4 188.  The same MFMA instruction and k order: the bits of k_gemm_pf, which keeps the epilogues of the layer-list models.
template <int EPI, int TM>
__global__ void __launch_bounds__(256, 1) k_gemm_pf_wide(PfGemmParams p, int mt, int tiles) {
    using G = GemmTiles<TM, true>;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[G::LDS];
    // Bands (TileOrder) from 13 row tiles on: 2929 rows, gate | up 252 -> 244 us, q|k|v 98 -> 86, o and down 98 -> 96, the pass 19.4 -> 18.8 ms; with fewer, one band holds every row tile and
    // W passes once (1030 rows in bands of 8: 11.1 ms, in one 10.9)
    const int band = mt > 12 ? (TM >= 6 ? 6 : 8) : mt;
    const TileOrder order{mt, tiles / mt};
    const int xcd = blockIdx.x & 7, lo = (int)((int64_t)tiles * xcd / 8), hi = (int)((int64_t)tiles * (xcd + 1) / 8), first = lo + (blockIdx.x >> 3);
    if (first >= hi) return;
    const int NT = p.N >> 4, KT = p.K >> 5, ldx = EPI == PF_ROWS_BF16 ? p.ex.ldx : p.K;
    int mr, nr;                                             // of the tile being requested
    G::run(lds, p.K, first, gridDim.x >> 3, hi,
           [&](int t, const bf16_t*& W, const bf16_t*& X) { order.at(band, t, mr, nr); W = p.Wp; X = p.X; },
           [&](int, int q, int lane) { return ((uint32_t)min(nr * (G::BN / 16) + (q >> 1), NT - 1) * KT + (q & 1)) * 512u + lane * 8; },
           [&](int, int r) { return (uint32_t)min(mr * G::BM + r, p.M - 1) * ldx; },
           [&](int t, const f32x4_t (&acc)[G::TN][TM]) {
               int mi, ni;
               order.at(band, t, mi, ni);
               int lane = threadIdx.x & 63;
               asm volatile("" : "+v"(lane));
               const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
               if constexpr (EPI == PF_RESID) {            // one row of tiles at a time, its residuals requested a row ahead (a wave has no other to wait with)
                   const int nb = ni * G::BN + (wave >> 1) * 128 + (lane >> 4) * 4, mb = mi * G::BM + (wave & 1) * TM * 16 + (lane & 15);
                   bf16_t* h = reinterpret_cast<bf16_t*>(p.C);
                   uint2 r[2][G::TN];
                   auto residual = [&](int j, uint2 (&o)[G::TN]) {
                       const bf16_t* row = h + (size_t)min(mb + j * 16, p.M - 1) * p.N;
#pragma unroll
                       for (int i = 0; i < G::TN; ++i) o[i] = *reinterpret_cast<const uint2*>(row + min(nb + i * 16, p.N - 4));
                   };
                   residual(0, r[0]);
#pragma unroll
                   for (int j = 0; j < TM; ++j) {
                       if (j + 1 < TM) residual(j + 1, r[(j + 1) & 1]);
                       __builtin_amdgcn_sched_barrier(0);
                       const int m = mb + j * 16;
#pragma unroll
                       for (int i = 0; i < G::TN; ++i) {
                           uint2& o = r[j & 1][i];
                           const float hv[4] = {__uint_as_float(o.x << 16), __uint_as_float(o.x & 0xffff0000u), __uint_as_float(o.y << 16), __uint_as_float(o.y & 0xffff0000u)};
                           uint16_t v[4];
#pragma unroll
                           for (int e = 0; e < 4; ++e) v[e] = f32_to_bf16(hv[e] + bf16_round_f32(acc[i][j][e]));       // h = T(h + T(x W^T))
                           o = make_uint2((uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16));
                           asm volatile("" : "+v"(o.x), "+v"(o.y));          // (not inside the branch below: a wait there waits for every store before it)
                       }
#pragma unroll
                       for (int i = 0; i < G::TN; ++i)
                           if (m < p.M && nb + i * 16 < p.N) *reinterpret_cast<uint2*>(h + (size_t)m * p.N + nb + i * 16) = r[j & 1][i];
                   }
                   return;
               }
               pf_epilogue<EPI, G::TN, TM>(p, acc, ni * (G::BN / 16) + (wave >> 1) * G::TN, mi * G::BM + (wave & 1) * TM * 16, lane);
           });
}
template <int EPI>
static bool launch_gemm_pf_wide(const PfGemmParams& p, hipStream_t s) {
    const int64_t ldx = EPI == PF_ROWS_BF16 ? p.ex.ldx : p.K;
    // (32-bit byte offsets; three k-steps at least fill the ring)
    if (p.K < 3 * PF_BK || (EPI == PF_ROWS_BF16 && p.ex.xrow) || (int64_t)p.N * p.K >= (1ll << 31) || (int64_t)p.M * ldx >= (1ll << 31)) return false;
    const int nt = cdiv(p.N, 256);
    int best = 0;
    double least = 0;
    for (int tm = 4; tm <= 6; ++tm) {                      // rounds of 256 blocks, each as long as its tiles are high and a little
        const double cost = cdiv(nt * cdiv(p.M, 32 * tm), 256) * (tm + 0.4);
        if (!best || cost < least) { best = tm; least = cost; }
    }
    // A block fills its ring and drains its last tile alone on its compute unit; k_gemm_pf has two, and is faster where K is short and its blocks are all there at
    // once, or in one and a half rounds against two.  us, k_gemm_pf / here: gate | up (N = 6144) K = 1024, 300 rows (144 blocks) 15 / 17, 1200 (480) 20 / 21, 1536
    // (576; 240 tiles) 31 / 25, 2048 (768; 384) 34 / 37; q|k|v (N = 4096) K = 1024, 600 rows 14 / 17, 2048 22 / 23, 2400 33 / 26; K = 512 (N = 4096), 900 rows 11 / 14, 3200
    // (800; 400) 23 / 25; K = 1536: N = 2048, 1200 rows (160) 24 / 26, 2816 (352) 29 / 27, N = 17920, 384 (420) 30 / 29, 608 (700; 350) 49 / 52; K = 2048, N = 1024, 1500 rows
    // (96) 32 / 31, N = 2048, 1800 (240) 35 / 35, 2816 40 / 36
    const int nx = cdiv(p.N, PF_BN), blocks = (nx >= 16 ? (int)round_up(nx, 8) : nx) * cdiv(p.M, PF_BM), rounds = cdiv(nt * cdiv(p.M, 32 * best), 256);
    if (p.K <= 1536 && (blocks <= (p.K <= 1024 ? 512 : 256) || (rounds > 1 && blocks <= (p.K <= 512 ? 1024 : 768)))) return false;
    auto go = [&](auto tag) {
        constexpr int TM = decltype(tag)::value;
        const int mt = cdiv(p.M, 32 * TM), tiles = mt * nt;
        hipLaunchKernelGGL((k_gemm_pf_wide<EPI, TM>), dim3(std::min((int)round_up(tiles, 8), 256)), dim3(256), 0, s, p, mt, tiles);
    };
    if (best == 4) go(std::integral_constant<int, 4>{});
    else if (best == 5) go(std::integral_constant<int, 5>{});
    else go(std::integral_constant<int, 6>{});
    return true;
}

// Few rows: k_gemm_pf waits 0.6 us for each of its 48 - 128 k-steps, and a short prompt's 24 - 128 tiles of 128 x 128 leave most of the chip idle meanwhile.
// Tiles of 32 rows x 32 columns (gate | up: 64, the pairs of a wave) on two waves, with a ring of NBUF k-steps in LDS requested ahead under counted waits: bound
// by the weights' way from memory.  The same MFMA instruction and k order: the bits of k_gemm_pf.  Orpheus-3B, us per launch, k_gemm_pf / here: 24 rows:
// o and down 81 / 17, q|k|v 44 / 12, gate | up 48 / 20; 60 rows: 83 / 17, 45 / 18, 49 / 35; 120 rows: 88 / 30, 50 / 26, 54 / 64.
// (The ring on 128 x 128 tiles: 79 for 83 us with o and down at 1024 rows, 83 for 51 with q|k|v.)
template <int EPI, int TN, int NBUF>
__global__ void __launch_bounds__(128) k_gemm_pf_ring(PfGemmParams p) {
    constexpr int WN = 2, WM = 1, TM = 2, NW = WN * WM, BN = WN * TN * 16, BM = WM * TM * 16, QW = WN * TN * 2 / NW, QX = WM * TM * 2 / NW, NQ = QW + QX;   // DMA instructions per wave and k-step
    constexpr int WB = WN * TN * 2048, STEP = WB + WM * TM * 2048;                                                        // bytes
    static_assert((NBUF - 2) * NQ <= 63 && QW * NW == WN * TN * 2 && QX * NW == WM * TM * 2, "vmcnt; whole DMA instructions");
    __shared__ __attribute__((aligned(1024))) unsigned char ring[NBUF * STEP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave / WM, wm = wave % WM;
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM, NT = p.N >> 4, KT = p.K >> 5, KS = p.K / PF_BK;
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const bf16_t *wsrc[QW], *xsrc[QX];                  // the staging of k_gemm_pf: W fragments as they are, X rows with swizzled 16-byte pieces
#pragma unroll
    for (int q = 0; q < QW; ++q) {
        const int f = wave * QW + q;
        wsrc[q] = p.Wp + ((size_t)min((n0 >> 4) + (f >> 1), NT - 1) * KT + (f & 1)) * 512 + lane * 8;
    }
#pragma unroll
    for (int q = 0; q < QX; ++q) {
        const int r = (wave * QX + q) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7), xm = min(m0 + r, p.M - 1);
        if constexpr (EPI == PF_ROWS_BF16) xsrc[q] = p.X + (size_t)(p.ex.xrow ? p.ex.xrow[xm] : xm) * p.ex.ldx + chunk * 8;
        else xsrc[q] = p.X + (size_t)xm * p.K + chunk * 8;
    }
    auto stage = [&](int buf, int ks) {
        unsigned char* l = ring + buf * STEP;
#pragma unroll
        for (int q = 0; q < QW; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wsrc[q] + (size_t)ks * 1024),
                                             (__attribute__((address_space(3))) void*)(l + (wave * QW + q) * 1024), 16, 0, 0);
#pragma unroll
        for (int q = 0; q < QX; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xsrc[q] + ks * PF_BK),
                                             (__attribute__((address_space(3))) void*)(l + WB + (wave * QX + q) * 1024), 16, 0, 0);
    };
    const int sw = (lane >> 1) & 7;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)ring;
    const uint32_t wa = base + wn * TN * 2048 + lane * 16, xa = base + WB + wm * TM * 2048 + (lane & 15) * 128;
    const uint32_t x0 = xa + ((lane >> 4) ^ sw) * 16, x1 = xa + ((4 + (lane >> 4)) ^ sw) * 16;
    for (int i = 0; i < NBUF - 1; ++i) stage(i, min(i, KS - 1));
    int rd = 0, wr = NBUF - 1;
    for (int ks = 0; ks < KS; ++ks) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * NQ) : "memory");      // this wave's part of k-step ks has landed
        __builtin_amdgcn_s_barrier();                                               // everybody's; the slot read one step ago is free
        const uint32_t o = rd * STEP;
        bf16x8_t a[2][TN], b[2][TM];
        // fragment reads and their wait in one block: behind an LDS-DMA the compiler would wait for every load in flight (see k_gemm_big3)
        if constexpr (TN == 1)
            asm volatile("ds_read_b128 %0, %6\n ds_read_b128 %1, %6 offset:1024\n ds_read_b128 %2, %7\n ds_read_b128 %3, %7 offset:2048\n"
                         "ds_read_b128 %4, %8\n ds_read_b128 %5, %8 offset:2048\n s_waitcnt lgkmcnt(0)"
                         : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
                         : "v"(wa + o), "v"(x0 + o), "v"(x1 + o) : "memory");
        else
            asm volatile("ds_read_b128 %0, %8\n ds_read_b128 %1, %8 offset:1024\n ds_read_b128 %2, %8 offset:2048\n ds_read_b128 %3, %8 offset:3072\n"
                         "ds_read_b128 %4, %9\n ds_read_b128 %5, %9 offset:2048\n ds_read_b128 %6, %10\n ds_read_b128 %7, %10 offset:2048\n s_waitcnt lgkmcnt(0)"
                         : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[0][TN - 1]), "=&v"(a[1][TN - 1]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
                         : "v"(wa + o), "v"(x0 + o), "v"(x1 + o) : "memory");
        stage(wr, min(ks + NBUF - 1, KS - 1));                                      // (past the end: the last step again, never read)
        rd = rd + 1 == NBUF ? 0 : rd + 1;
        wr = wr + 1 == NBUF ? 0 : wr + 1;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][i], b[kk][j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                // (no DMA into the LDS of a block that has ended)
    pf_epilogue<EPI, TN, TM>(p, acc, (n0 >> 4) + wn * TN, m0 + wm * TM * 16, lane);
}

// ---- prompt GEMMs on 8- / 4-bit codes (layouts and arithmetic of lm_qgemm.hip: y = sum over groups of 64 of scale * sum(q x) + bias * sum(x), codes exact in
// bf16, float32 sums).  The decode step's kernels take 64 rows a launch and read the weights again for each; here a block of 64 TM/2 x 64 TN/2 outputs unpacks a
// code once for all its rows, into the fragment image that k_gemm_pf reads.  A k-step is a scale group: X by LDS-DMA and codes and scales through registers one step
// ahead, one barrier.  Bound: a group costs an output a product, an FMA and an addition beside its 64 products - VALU above matrix pipe, two blocks a compute unit
// share both.  (Two FMAs into one chain of sums are 10 % faster at 128 x 128 - gate | up of 3216 rows 583 us, 641 here - but then a prompt's bits depend on the
// other prompts of its call, which decide between the kernels.)
// Prompt pass of Orpheus-3B at 8 bits, ms, slices of 64 rows / here: 804 rows 33.6 / 16.2, 3202 129 / 46.6; here, the kernels of 176 rows: 6.4 (8.2 with one team a block).
__device__ __forceinline__ uint4 pf_codes(uint2 w) {
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t v = e < 2 ? w.x >> (16 * e) : w.y >> (16 * (e - 2));
        o[e] = (uint32_t)f32_to_bf16((float)(v & 0xffu)) | ((uint32_t)f32_to_bf16((float)((v >> 8) & 0xffu)) << 16);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}
__device__ __forceinline__ uint4 pf_codes(uint32_t w) {
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = (uint32_t)f32_to_bf16((float)((w >> (8 * e)) & 0xfu)) | ((uint32_t)f32_to_bf16((float)((w >> (8 * e + 4)) & 0xfu)) << 16);
    return make_uint4(o[0], o[1], o[2], o[3]);
}
template <int BITS> struct PfCode { typedef uint2 type; };
template <> struct PfCode<4> { typedef uint32_t type; };

// Q: teams of four waves, each with a quarter of the groups (4) or all of them (1)
template <int EPI, int TN, int TM, int BITS, int Q>
__global__ void __launch_bounds__(256 * Q, Q == 1 ? 2 : 4) k_gemm_pf_codes(PfGemmParams p, const void* __restrict__ Qp, const bf16_t* __restrict__ SB) {
    typedef typename PfCode<BITS>::type WT;
    constexpr int BN = 32 * TN, BM = 32 * TM, HELD = TN == 4 ? 2 : 0;
    __shared__ f32x4_t held[HELD ? HELD : 1][256];
    static_assert(Q == 1 || (Q == 4 && !HELD), "one team, or one a quarter");
    __shared__ __attribute__((aligned(1024))) bf16_t Wt[Q][2][BN * PF_BK];
    __shared__ __attribute__((aligned(1024))) bf16_t Xt[Q][2][BM * PF_BK];
    const int tid = Q == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int team = Q == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    bf16_t (&Ws)[2][BN * PF_BK] = Wt[team];
    bf16_t (&Xs)[2][BM * PF_BK] = Xt[team];
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
    if (n0 >= p.N) return;                              // (padding of the grid, see launch_gemm_pf)
    const int wn = wave >> 1, wm = wave & 1, NT = p.N >> 4, KT = p.K >> 5, G = p.K / PF_BK;
    const int ga = G * team / Q, gb = G * (team + 1) / Q, steps = (G + Q - 1) / Q;         // (ceil(G / 4): the longest quarter)
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // a wave stages TN of the block's 4 TN weight fragments (2 TN n-tiles x 2 k-tiles) and TM KB of X (k_gemm_pf's image); it reads the scales of its own n-tiles
    // (bases per wave in scalar registers, 32-bit offsets per lane: the totals need the others)
    const WT* wsrc[TN];
    const uint2* sbp[TN];
    uint32_t xoff[TM];
#pragma unroll
    for (int q = 0; q < TN; ++q) {
        const int f = wave * TN + q;
        wsrc[q] = reinterpret_cast<const WT*>(Qp) + ((size_t)min((n0 >> 4) + (f >> 1), NT - 1) * KT + (f & 1)) * 64;
        sbp[q] = reinterpret_cast<const uint2*>(SB) + (size_t)min((n0 >> 4) + wn * TN + q, NT - 1) * G * 8;
    }
#pragma unroll
    for (int q = 0; q < TM; ++q) {
        const int r = (wave * TM + q) * 8 + (lane >> 3);
        xoff[q] = ((uint32_t)min(m0 + r, p.M - 1) * p.K + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2;
    }
    const uint32_t sl = lane >> 4;
    WT w[TN];
    uint2 sb[TN][2];
    auto loadW = [&](int g) {                           // (groups past the end: the last one again, never multiplied)
#pragma unroll
        for (int q = 0; q < TN; ++q) w[q] = (wsrc[q] + (size_t)min(g, G - 1) * 128)[(uint32_t)lane];
    };
    auto loadS = [&](int g, int q) {
        const uint2* o = sbp[q] + (size_t)min(g, G - 1) * 8;
        sb[q][0] = o[sl]; sb[q][1] = o[sl + 4];
    };
    auto putW = [&](int buf) {
#pragma unroll
        for (int q = 0; q < TN; ++q) *reinterpret_cast<uint4*>(&Ws[buf][(wave * TN + q) * 512 + lane * 8]) = pf_codes(w[q]);
    };
    auto stageX = [&](int buf, int g) {
#pragma unroll
        for (int q = 0; q < TM; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(reinterpret_cast<const unsigned char*>(p.X + (size_t)min(g, G - 1) * PF_BK) + xoff[q]),
                                             (__attribute__((address_space(3))) void*)&Xs[buf][(wave * TM + q) * 8 * PF_BK], 16, 0, 0);
    };
    bf16x8_t ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (short)0x3F80;
    const f32x4_t zero = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // A row is to have the bits that k_gemm_skinny_q gives it: its four waves sum a quarter of the groups each, the quarters are added in order.  The total of the
    // large tile's last HELD products waits in LDS: the registers hold 248 values beside it
    f32x4_t tot[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) tot[i][j] = zero;
    auto close = [&](bool first) {                      // (0 + p0 is p0: a sum that starts at 0 is never -0)
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int h = i * TM + j - (TN * TM - HELD);
                f32x4_t t = h < 0 ? tot[i][j] : first ? zero : held[h < 0 ? 0 : h][tid];
#pragma unroll
                for (int e = 0; e < 4; ++e) t[e] += acc[i][j][e];
                acc[i][j] = zero;
                if (h < 0) tot[i][j] = t;
                else held[h < 0 ? 0 : h][tid] = t;
            }
    };
    int part = 1;                                       // the quarter of the groups that begins next
    const int sw = (lane >> 1) & 7;
    loadW(ga);
    putW(0);
    loadW(ga + 1);
#pragma unroll
    for (int q = 0; q < TN; ++q) loadS(ga, q);
    stageX(0, ga);
    for (int g = ga, st = 0, buf = 0; st < steps; ++st, ++g, buf ^= 1) {
        __syncthreads();                                // X and codes of this step are in LDS, the codes of the next and the scales of this one in registers
        bf16x8_t a[2][TN], b[2][TM];                    // all fragment reads first, then the next DMA (see k_gemm_pf)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int pos = ((kk * 4 + (lane >> 4)) ^ sw) * 8;
#pragma unroll
            for (int i = 0; i < TN; ++i) a[kk][i] = *reinterpret_cast<const bf16x8_t*>(&Ws[buf][((wn * TN + i) * 2 + kk) * 512 + lane * 8]);
#pragma unroll
            for (int j = 0; j < TM; ++j) b[kk][j] = *reinterpret_cast<const bf16x8_t*>(&Xs[buf][(wm * TM * 16 + j * 16 + (lane & 15)) * PF_BK + pos]);
        }
        const bool more = st + 1 < steps;
        if (more) putW(buf ^ 1);                        // (the other buffer: read by everybody before this step's barrier)
        __builtin_amdgcn_sched_barrier(0);
        loadW(g + 2);
        if (more) stageX(buf ^ 1, g + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (Q > 1 && g >= gb) continue;                 // (a shorter quarter: the barriers of the others)
        if (Q == 1 && part < 4 && g == G * part / 4) {
            close(part == 1);
            do ++part; while (part < 4 && G * part / 4 == g);
        }
        float sx[TM];                               // (the rows of a tile of ones are one row)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            f32x4_t t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[0][j], zero, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[1][j], t, 0, 0, 0);
            sx[j] = t[0];
        }
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const uint2 s0 = sb[i][0], b0 = sb[i][1];
            const float sc[4] = {__uint_as_float(s0.x << 16), __uint_as_float(s0.x & 0xffff0000u), __uint_as_float(s0.y << 16), __uint_as_float(s0.y & 0xffff0000u)};
            const float bi[4] = {__uint_as_float(b0.x << 16), __uint_as_float(b0.x & 0xffff0000u), __uint_as_float(b0.y << 16), __uint_as_float(b0.y & 0xffff0000u)};
#pragma unroll
            for (int j0 = 0; j0 < TM; j0 += 2) {
                f32x4_t ag[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) ag[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0][i], b[0][j0 + j], zero, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j) ag[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1][i], b[1][j0 + j], ag[j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j0 + j][e] += fmaf(sc[e], ag[j][e], bi[e] * sx[j0 + j]);
            }
            loadS(g + 1, i);               // (the next step's, into the registers just read)
        }
    }
    if constexpr (Q > 1) {                              // the quarters in order: those of the others through LDS
        f32x4_t (*sums)[TN * TM][256] = reinterpret_cast<f32x4_t (*)[TN * TM][256]>(&Wt[0][0][0]);
        static_assert((Q - 1) * TN * TM * 256 * sizeof(f32x4_t) <= sizeof(Wt), "the sums fit where the codes were");
        __syncthreads();
        if (team)
#pragma unroll
            for (int i = 0; i < TN * TM; ++i) sums[team - 1][i][tid] = acc[i / TM][i % TM];
        __syncthreads();
        if (team) return;
#pragma unroll
        for (int i = 0; i < TN * TM; ++i) {
            f32x4_t t = acc[i / TM][i % TM];
#pragma unroll
            for (int w2 = 0; w2 < Q - 1; ++w2)
#pragma unroll
                for (int e = 0; e < 4; ++e) t[e] += sums[w2][i][tid][e];
            tot[i / TM][i % TM] = t;
        }
    } else
        close(false);
#pragma unroll
    for (int h = 0; h < HELD; ++h) tot[(TN * TM - HELD + h) / TM][(TN * TM - HELD + h) % TM] = held[h][tid];
    pf_epilogue<EPI, TN, TM>(p, tot, (n0 >> 4) + wn * TN, m0 + wm * TM * 16, lane);
}
void launch_gemm_pf_codes(int epi, int bits, const bf16_t* X, const void* Qp, const bf16_t* SB, void* C, int M, int N, int K, hipStream_t s) {
    MIS_REQUIRE(K % PF_BK == 0 && K >= PF_BK && N % 16 == 0 && M >= 1 && (bits == 8 || bits == 4) && (epi != PF_SILU || N % 32 == 0) && (int64_t)M * K < (1ll << 31),
                MIS_ERR_GENERATION_FAILED, "prefill GEMM on codes: bad shape");
    PfGemmParams p{X, nullptr, C, M, N, K, PfExtra()};
    auto go = [&](auto e, auto t, auto q, auto b) {
        constexpr int E = decltype(e)::value, T = decltype(t)::value, Q = decltype(q)::value, B = decltype(b)::value;
        const int nx = cdiv(N, 32 * T);
        hipLaunchKernelGGL((k_gemm_pf_codes<E, T, T, B, Q>), dim3(nx >= 16 ? (int)round_up(nx, 8) : nx, cdiv(M, 32 * T)), dim3(256 * Q), 0, s, p, Qp, SB);
    };
    auto tile = [&](auto e, auto b) {
        // Up to 512 tiles of 64 x 64: a team of waves for each quarter of K, one block a compute unit (131 KB).  With one team and four groups a step (two from 257 tiles on) a
        // wave a SIMD waited for each step's loads, fragments and conversions in turn.  Orpheus-3B, 8 bits, us, one team / four: 176 rows o (144 tiles) 36 / 23, down 89 / 54,
        // q|k|v (240) 38 / 24; 256 rows q|k|v (320) 46 / 41; 400 rows o (336) 45 / 42.  More tiles: 800 rows o (624) 57 / 60, q|k|v (1040) 73 / 79.  128 x 128: o 1632 rows
        // (312 blocks) 107, gate | up 3216 (3328) 641: 500 TFLOP/s.  Narrower, a prompt pass of four layers in us, teams up to 256 tiles / up to 512: width 1024 (q|k|v 320 - 512
        // tiles) 257 rows 626 / 618, 512 707 / 702; 2048 128 rows (gate | up 384) 690 / 663, 257 (q|k|v 320) 966 / 927; at 4 bits 257 986 / 974, 512 1069 / 1053
        const int64_t nb = (int64_t)cdiv(N, 64) * cdiv(M, 64);
        if ((int64_t)cdiv(N, 128) * cdiv(M, 128) >= 256) go(e, std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{}, b);
        else if (nb > 512) go(e, std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{}, b);
        else go(e, std::integral_constant<int, 2>{}, std::integral_constant<int, 4>{}, b);
    };
    auto width = [&](auto e) {
        if (bits == 8) tile(e, std::integral_constant<int, 8>{});
        else tile(e, std::integral_constant<int, 4>{});
    };
    if (epi == PF_F32) width(std::integral_constant<int, PF_F32>{});
    else if (epi == PF_RESID) width(std::integral_constant<int, PF_RESID>{});
    else if (epi == PF_SILU) width(std::integral_constant<int, PF_SILU>{});
    else throw MisError(MIS_ERR_GENERATION_FAILED, "unknown prefill GEMM epilogue");
    HIP_CHECK(hipGetLastError());
}

void launch_gemm_pf(int epi, const bf16_t* X, const bf16_t* Wp, void* C, int M, int N, int K, hipStream_t s, const PfExtra& ex) {
    MIS_REQUIRE(K % PF_BK == 0 && K >= 2 * PF_BK && N % 16 == 0 && M >= 1, MIS_ERR_GENERATION_FAILED, "prefill GEMM: K must be a multiple of 64");
    MIS_REQUIRE((epi != PF_SILU && epi != PF_SWIGLU) || N % 32 == 0, MIS_ERR_GENERATION_FAILED, "prefill GEMM: gate / up tiles come in pairs");
    MIS_REQUIRE(epi < PF_SPLIT_RELU2 || epi == PF_SWIGLU || (ex.ldc % 4 == 0 && (epi != PF_ROWS_BF16 || ex.ldx % 8 == 0)), MIS_ERR_GENERATION_FAILED,
                "prefill GEMM: bad row strides");
    PfGemmParams p{X, Wp, C, M, N, K, ex};
    // Few blocks of the small tile (the larger one reads a weight tile once per 128 rows, not per 32).  o and down at 240 / 400 rows (768 / 1248 blocks): 44 / 71
    // against 85 / 82 us; q|k|v at 240 / 400 (1280 / 2080): 43 / 70 against 48 / 45; gate | up at 60 / 120 (512 / 1024): 35 / 64 against 49 / 54.
    auto few = [&](auto e) {
        constexpr int E = decltype(e)::value, TN = E == PF_SILU ? 2 : 1;
        if ((int64_t)cdiv(N, 32 * TN) * cdiv(M, 32) > (TN == 2 ? 512 : 1280)) return false;
        hipLaunchKernelGGL((k_gemm_pf_ring<E, TN, TN == 2 ? 12 : 16>), dim3(cdiv(N, 32 * TN), cdiv(M, 32)), dim3(128), 0, s, p);
        return true;
    };
    if (epi == PF_F32 && few(std::integral_constant<int, PF_F32>{})) return;
    if (epi == PF_RESID && few(std::integral_constant<int, PF_RESID>{})) return;
    if (epi == PF_SILU && few(std::integral_constant<int, PF_SILU>{})) return;
    if (epi == PF_ROWS_BF16 && few(std::integral_constant<int, PF_ROWS_BF16>{})) return;
    if (epi == PF_RESID && launch_gemm_pf_wide<PF_RESID>(p, s)) return;
    if (epi == PF_SILU && launch_gemm_pf_wide<PF_SILU>(p, s)) return;
    if (epi == PF_ROWS_BF16 && launch_gemm_pf_wide<PF_ROWS_BF16>(p, s)) return;
    // column tiles rounded up to the 8 XCDs: blocks are dealt to the XCDs by linear id, so that every row of tiles finds its weight tiles in the
    // L2 that held them for the row before
    const int nx = cdiv(N, PF_BN);
    dim3 grid(nx >= 16 ? (int)round_up(nx, 8) : nx, cdiv(M, PF_BM)), block(256);
    if (epi == PF_F32) hipLaunchKernelGGL((k_gemm_pf<PF_F32>), grid, block, 0, s, p);
    else if (epi == PF_RESID) hipLaunchKernelGGL((k_gemm_pf<PF_RESID>), grid, block, 0, s, p);
    else if (epi == PF_SILU) hipLaunchKernelGGL((k_gemm_pf<PF_SILU>), grid, block, 0, s, p);
    else if (epi == PF_SPLIT_RELU2) hipLaunchKernelGGL((k_gemm_pf<PF_SPLIT_RELU2>), grid, block, 0, s, p);
    else if (epi == PF_SCALED_ADD) hipLaunchKernelGGL((k_gemm_pf<PF_SCALED_ADD>), grid, block, 0, s, p);
    else if (epi == PF_ROWS_BF16) hipLaunchKernelGGL((k_gemm_pf<PF_ROWS_BF16>), grid, block, 0, s, p);
    else if (epi == PF_SOFTCAP) hipLaunchKernelGGL((k_gemm_pf<PF_SOFTCAP>), grid, block, 0, s, p);
    else if (epi == PF_SWIGLU) hipLaunchKernelGGL((k_gemm_pf<PF_SWIGLU>), grid, block, 0, s, p);
    else if (epi == PF_ACT_ROWS) hipLaunchKernelGGL((k_gemm_pf<PF_ACT_ROWS>), grid, block, 0, s, p);
    else throw MisError(MIS_ERR_GENERATION_FAILED, "unknown prefill GEMM epilogue");
}
void launch_pf_embed_rmsnorm(const bf16_t* emb, const int32_t* prompt, const int32_t* lens, int Lmax, int t0, int Tc, int batch, int Mpad, int vocab,
                             const bf16_t* wnorm, bf16_t* h, bf16_t* x, int32_t* pos_tab, uint8_t* act_tab, int rows, int d, float eps, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_embed_rmsnorm, dim3(rows), dim3(256), 0, s, emb, prompt, lens, Lmax, t0, Tc, batch, Mpad, vocab, wnorm, h, x, pos_tab,
                       act_tab, d, eps);
}
void launch_pf_rows_rmsnorm(const bf16_t* rows, int src_rows, const int32_t* lens, int Lmax, int t0, int Tc, int batch, int Mpad, const bf16_t* wnorm,
                            bf16_t* h, bf16_t* x, int32_t* pos_tab, uint8_t* act_tab, int n_rows, int d, float eps, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_rows_rmsnorm, dim3(n_rows), dim3(256), 0, s, rows, src_rows, lens, Lmax, t0, Tc, batch, Mpad, wnorm, h, x, pos_tab, act_tab, d, eps);
}
void launch_pf_rmsnorm(const bf16_t* h, const bf16_t* wnorm, bf16_t* x, int rows, int d, float eps, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_rmsnorm, dim3(rows), dim3(256), 0, s, h, wnorm, x, d, eps);
}
// h = T(h + T(part)): the residual add behind a GEMM that wrote float32 sums (quantised roles run the decode step's code-streaming
// kernel on 64-row chunks; same rounding points as the PF_RESID epilogue and the decode step's glue)
__global__ void k_pf_add_resid(bf16_t* __restrict__ h, const float* __restrict__ part, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) h[i] = f32_to_bf16(bf16_to_f32(h[i]) + bf16_round_f32(part[i]));
}
void launch_pf_add_resid(bf16_t* h, const float* part, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_add_resid, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, h, part, n);
}
void launch_pf_pack_last(const bf16_t* rows, const int32_t* lens, int Lmax, int t0, int Tc, int batch, bf16_t* xpk, int Mpad, int d, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_pack_last, dim3(Mpad), dim3(256), 0, s, rows, lens, Lmax, t0, Tc, batch, xpk, d, Mpad / 16);
}
void launch_pf_pack_rows(const bf16_t* rows, bf16_t* xpk, int Mpad, int d, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_pack_rows, dim3(Mpad), dim3(256), 0, s, rows, xpk, d, Mpad / 16);
}

// ============================================================================ causal attention of a chunk of positions
//
// Two launches per layer.  k_pf_rope_append rounds q|k|v to bf16, applies the per-head norm (where the model has one) and the rotation, writes the
// queries as bf16 rows and the keys / values into the decode step's tiled caches (whole 16-byte pieces; one block = the positions of one 32-key tile
// of one kv head of one sequence).  k_pf_attn then walks the cache tiles: the G query heads of a kv head times its positions are ONE list of queries
// (query n = position n / G, head n % G), a block takes 32 of them per wave, stages every 32-key tile's K and V images once through LDS (two buffers,
// the next tile requested before this one is multiplied) and uses each fragment for both of a wave's groups of 16 queries.  A tile above a
// wave's last position is skipped, only tiles that reach a wave's positions are masked, and the output is rescaled only when some maximum moved.
// A query's sums run over the tiles 0, 1, 2, ... whatever block, chunk or batch it is part of: the same bits in every arrangement.
// P enters P.V as bf16 hi + lo (probabilities keep float32 accuracy), like the decode step.
// Measured (8 rows x 450 positions, 24 / 8 heads x 128): 59 us attention + 25 us rope / append per layer; the decode kernel with one block per (position,
// kv head), which stood here before, streamed every query's whole cache for itself: 766 us.  Bound now: the softmax's VALU work and one barrier a tile.
// float32 q|k|v rows would cost another 37 MB written and read per layer: the projection rounds them, which is the first thing the attention did.
struct PfAttnDev {
    const void* qkv; int Nqkv;
    bf16_t *q, *kc, *vc, *out;
    const int32_t* lens;
    int Lmax, t0, tc, H, Hkv, Smax;
    const float *rope_cos, *rope_sin;
    const bf16_t *qnorm_w, *knorm_w;
    float qk_eps, scale;
    int rope_in_dtype;
};
__device__ __forceinline__ void pf_load8(const float* src, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
    v[0] = bf16_round_f32(a.x); v[1] = bf16_round_f32(a.y); v[2] = bf16_round_f32(a.z); v[3] = bf16_round_f32(a.w);
    v[4] = bf16_round_f32(b.x); v[5] = bf16_round_f32(b.y); v[6] = bf16_round_f32(b.z); v[7] = bf16_round_f32(b.w);
}
__device__ __forceinline__ void pf_load8(const bf16_t* src, float (&v)[8]) {
    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(src);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_to_f32((bf16_t)a[e]);
}
template <int D, typename TIN>
__global__ void __launch_bounds__(256) k_pf_rope_append(PfAttnDev p) {
    constexpr int VT = D / 16;                                   // threads per head row: 8 dimensions and their 8 rotation partners each
    __shared__ __attribute__((aligned(16))) bf16_t vs[32][D + 8];
    const int b = blockIdx.z, kvh = blockIdx.y, tid = threadIdx.x;
    const PfSpan sp = pf_span(p.lens, b, p.Lmax, p.t0, p.tc);
    const int tile = (sp.lo >> 5) + blockIdx.x, p0 = max(tile * 32, sp.lo), p1 = min(tile * 32 + 32, sp.hi);
    if (p0 >= p1) return;
    const int G = p.H / p.Hkv;
    const TIN* qkv = reinterpret_cast<const TIN*>(p.qkv);
    bf16_t* kc = p.kc + ((size_t)(b * p.Hkv + kvh) * p.Smax) * D;
    bf16_t* vc = p.vc + ((size_t)(b * p.Hkv + kvh) * p.Smax) * D;
    for (int it = tid; it < (p1 - p0) * VT * 2; it += 256) {     // V rows -> LDS
        const int i = it / (VT * 2), c = it - i * (VT * 2), pos = p0 + i;
        const size_t row = sp.row0 + pos;
        float v[8];
        pf_load8(qkv + row * p.Nqkv + (size_t)(p.H + p.Hkv + kvh) * D + c * 8, v);
        bf16x8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (short)f32_to_bf16(v[e]);
        *reinterpret_cast<bf16x8_t*>(&vs[pos & 31][c * 8]) = o;
    }
    for (int it = tid; it < (p1 - p0) * (G + 1) * VT; it += 256) {
        const int j = it % VT, hr = it / VT, i = hr / (G + 1), hh = hr - i * (G + 1), pos = p0 + i;
        const size_t row = sp.row0 + pos;
        const int col = (hh < G ? kvh * G + hh : p.H + kvh) * D + j * 8;
        float x1[8], x2[8];
        pf_load8(qkv + row * p.Nqkv + col, x1);
        pf_load8(qkv + row * p.Nqkv + col + D / 2, x2);
        if (p.qnorm_w) {                                         // n = T(x rsqrt(mean x^2 + eps)), T(w n)
            float ss = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x1[e] * x1[e] + x2[e] * x2[e];
#pragma unroll
            for (int o = 1; o < VT; o <<= 1) ss += __shfl_xor(ss, o, 64);
            const float inv = 1.0f / sqrtf(ss / (float)D + p.qk_eps);
            const bf16_t* w = hh < G ? p.qnorm_w : p.knorm_w;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x1[e] = bf16_round_f32(bf16_to_f32(w[j * 8 + e]) * bf16_round_f32(x1[e] * inv));
                x2[e] = bf16_round_f32(bf16_to_f32(w[D / 2 + j * 8 + e]) * bf16_round_f32(x2[e] * inv));
            }
        }
        const float* ct = p.rope_cos + (size_t)pos * (D / 2) + j * 8;
        const float* st = p.rope_sin + (size_t)pos * (D / 2) + j * 8;
        bf16x8_t r1, r2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float c = ct[e], s = st[e];
            if (p.rope_in_dtype) {
                c = bf16_round_f32(c); s = bf16_round_f32(s);
                r1[e] = (short)f32_to_bf16(bf16_round_f32(x1[e] * c) + bf16_round_f32(-x2[e] * s));
                r2[e] = (short)f32_to_bf16(bf16_round_f32(x2[e] * c) + bf16_round_f32(x1[e] * s));
            } else {
                r1[e] = (short)f32_to_bf16(x1[e] * c - x2[e] * s);
                r2[e] = (short)f32_to_bf16(x1[e] * s + x2[e] * c);
            }
        }
        if (hh < G) {
            bf16_t* o = p.q + row * ((size_t)p.H * D) + col;
            *reinterpret_cast<bf16x8_t*>(o) = r1;
            *reinterpret_cast<bf16x8_t*>(o + D / 2) = r2;
        } else {                                                 // K tiling: fragment row `prow` of half `half` (lm_kernels.hip), 8 dimensions = one piece
            const int pr = pos & 31, prow = ((pr >> 3) << 2) | (pr & 3), half = (pr >> 2) & 1;
            bf16_t* o = kc + ((size_t)tile * 2 + half) * (D / 32) * 512 + prow * 8;
            const int d2 = D / 2 + j * 8;
            *reinterpret_cast<bf16x8_t*>(o + ((j >> 2) * 64 + ((j & 3) << 4)) * 8) = r1;
            *reinterpret_cast<bf16x8_t*>(o + ((d2 >> 5) * 64 + (((d2 & 31) >> 3) << 4)) * 8) = r2;
        }
    }
    __syncthreads();
    const int a0 = p0 & 31, a1 = a0 + (p1 - p0);                 // slots of the tile that this chunk fills
    for (int it = tid; it < 4 * D; it += 256) {                  // V tiling: piece (d, octet of keys)
        const int d = it & (D - 1), o = it / D;
        bf16_t* dst = vc + (((size_t)tile * (D / 16) + (d >> 4)) * 64 + (o << 4) + (d & 15)) * 8;
        if (o * 8 >= a0 && o * 8 + 8 <= a1) {
            bf16x8_t v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (short)vs[o * 8 + e][d];
            *reinterpret_cast<bf16x8_t*>(dst) = v;
        } else {
            for (int e = 0; e < 8; ++e)
                if (o * 8 + e >= a0 && o * 8 + e < a1) dst[e] = vs[o * 8 + e][d];
        }
    }
}

template <int D, int NW>
__global__ void __launch_bounds__(NW * 64) k_pf_attn(PfAttnDev p) {
    constexpr int IMG = 32 * D, PIECES = 2 * IMG / 8 / (NW * 64);    // bf16 elements of one K (or V) tile image; 16-byte pieces per thread
    static_assert(PIECES * NW * 64 * 8 == 2 * IMG, "whole pieces");
    __shared__ __attribute__((aligned(16))) bf16_t kv[2][2 * IMG];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = blockIdx.y, b = blockIdx.z, G = p.H / p.Hkv;
    const PfSpan sp = pf_span(p.lens, b, p.Lmax, p.t0, p.tc);
    const int nq = (sp.hi - sp.lo) * G;
    const int nb = (nq + 32 * NW - 1) / (32 * NW), blk = nb - 1 - (int)blockIdx.x;   // the longest blocks first
    if (blk < 0) return;
    const int n0 = blk * 32 * NW, w0 = n0 + wave * 32;
    const int j = lane & 15, g4 = lane >> 4;
    const int HD = p.H * D;
    bf16x8_t qf[2][D / 32];
    int qpos[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int n = min(w0 + 16 * g + j, nq - 1);                  // (queries past the list repeat the last one; never written)
        const int pos = sp.lo + n / G;
        qpos[g] = pos;
        const bf16_t* src = p.q + (size_t)(sp.row0 + pos) * HD + (size_t)(kvh * G + n % G) * D + g4 * 8;
#pragma unroll
        for (int c = 0; c < D / 32; ++c) qf[g][c] = *reinterpret_cast<const bf16x8_t*>(src + c * 32);
    }
    const int wlo = sp.lo + min(w0, nq - 1) / G, whi = w0 < nq ? sp.lo + min(w0 + 31, nq - 1) / G : -1;       // positions of the wave's queries
    const int n_tiles = (sp.lo + min(n0 + 32 * NW - 1, nq - 1) / G) / 32 + 1;
    const size_t base = ((size_t)(b * p.Hkv + kvh) * p.Smax) * D;
    const uint4* ksrc = reinterpret_cast<const uint4*>(p.kc + base);
    const uint4* vsrc = reinterpret_cast<const uint4*>(p.vc + base);
    uint4 st[PIECES];
    auto fetch = [&](int tile) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int pc = tid + i * NW * 64;                        // K image first, V image behind it
            st[i] = pc < IMG / 8 ? ksrc[(size_t)tile * (IMG / 8) + pc] : vsrc[(size_t)tile * (IMG / 8) + pc - IMG / 8];
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) *(reinterpret_cast<uint4*>(kv[buf]) + tid + i * NW * 64) = st[i];
    };
    fetch(0);
    put(0);
    __syncthreads();
    f32x4_t O[2][D / 16];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) O[g][dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.0f, 0.0f};
    auto tile_math = [&](int tile, const bf16_t* img, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        const int kb = tile * 32 + g4 * 8;
        const bf16x8_t* kf = reinterpret_cast<const bf16x8_t*>(img) + lane;
        const bf16x8_t* vf = reinterpret_cast<const bf16x8_t*>(img + IMG) + lane;
        f32x4_t S[2][2];
#pragma unroll
        for (int g = 0; g < 2; ++g) S[g][0] = S[g][1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
            const bf16x8_t a0 = kf[c * 64], a1 = kf[((D / 32) + c) * 64];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                S[g][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, qf[g][c], S[g][0], 0, 0, 0);
                S[g][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, qf[g][c], S[g][1], 0, 0, 0);
            }
        }
        bf16x8_t ph[2], pl[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {                                // lane (query j, group g4): scores of keys kb .. kb + 7
            float sc[8], mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = S[g][e >> 2][e & 3] * p.scale;
                if constexpr (MASKED) v = kb + e <= qpos[g] ? v : -INFINITY;
                sc[e] = v;
                mx = fmaxf(mx, v);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run[g], mx);                 // (tile 0 holds key 0, which every query sees: finite from there on)
            const float alpha = __expf(m_run[g] - m_new);
            float psum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pe = __expf(sc[e] - m_new);
                psum += pe;
                const bf16_t hi = f32_to_bf16(pe);
                ph[g][e] = (short)hi;
                pl[g][e] = (short)f32_to_bf16(pe - bf16_to_f32(hi));
            }
            l_run[g] = l_run[g] * alpha + psum;
            const bool moved = m_new != m_run[g];
            m_run[g] = m_new;
            if (__any(moved)) {                                      // (alpha = 1 for every query otherwise)
                float ar[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, g4 * 4 + r, 64);
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) O[g][dt][r] *= ar[r];
            }
        }
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            const bf16x8_t vb = vf[dt * 64];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                O[g][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph[g], vb, O[g][dt], 0, 0, 0);
                O[g][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[g], vb, O[g][dt], 0, 0, 0);
            }
        }
    };
    for (int tile = 0; tile < n_tiles; ++tile) {
        const bool more = tile + 1 < n_tiles;
        if (more) fetch(tile + 1);
        if (tile * 32 + 31 <= wlo) tile_math(tile, kv[tile & 1], std::false_type{});
        else if (tile * 32 <= whi) tile_math(tile, kv[tile & 1], std::true_type{});
        if (more) put((tile + 1) & 1);
        __syncthreads();
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        float l = l_run[g];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r) {                                // O[g][dt][r]: query g4 * 4 + r, dimension dt * 16 + j
            const float lr = __shfl(l, g4 * 4 + r, 64);
            const int n = w0 + 16 * g + g4 * 4 + r;
            if (n < nq) {
                bf16_t* o = p.out + (size_t)(sp.row0 + sp.lo + n / G) * HD + (size_t)(kvh * G + n % G) * D + j;
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt) o[dt * 16] = f32_to_bf16(O[g][dt][r] / lr);
            }
        }
    }
}

void launch_pf_attention(const PfAttn& a, hipStream_t s) {
    MIS_REQUIRE(a.D == 64 || a.D == 128, MIS_ERR_INVALID_INPUT, "head_dim must be 64 or 128");
    MIS_REQUIRE(a.H % a.Hkv == 0 && a.Smax % 32 == 0 && a.t0 + a.tc <= a.Smax && a.Nqkv == (a.H + 2 * a.Hkv) * a.D, MIS_ERR_GENERATION_FAILED,
                "prompt attention: bad dimensions");
    MIS_REQUIRE((((uintptr_t)a.qkv | (uintptr_t)a.q | (uintptr_t)a.kcache | (uintptr_t)a.vcache) & 15) == 0, MIS_ERR_GENERATION_FAILED, "prompt attention: misaligned buffers");
    PfAttnDev p{a.qkv, a.Nqkv, a.q, a.kcache, a.vcache, a.out, a.lens, a.Lmax, a.t0, a.tc, a.H, a.Hkv, a.Smax, a.rope_cos, a.rope_sin, a.qnorm_w, a.knorm_w,
                a.qk_eps, a.scale, a.rope_in_dtype};
    const dim3 ga(a.tc / 32 + 2, a.Hkv, a.batch);                    // 32-key tiles that tc consecutive positions can touch
    const int nq = a.tc * (a.H / a.Hkv);
    // 256 queries a block share each staged tile where that still gives every compute unit a block; 128 otherwise
    const bool wide = (long)cdiv(nq, 256) * a.Hkv * a.batch >= 256;
    const dim3 gt(cdiv(nq, wide ? 256 : 128), a.Hkv, a.batch);
    auto go = [&](auto tag) {
        constexpr int D = decltype(tag)::value;
        if (a.qkv_f32) hipLaunchKernelGGL((k_pf_rope_append<D, float>), ga, dim3(256), 0, s, p);
        else hipLaunchKernelGGL((k_pf_rope_append<D, bf16_t>), ga, dim3(256), 0, s, p);
        if (wide) hipLaunchKernelGGL((k_pf_attn<D, 8>), gt, dim3(512), 0, s, p);
        else hipLaunchKernelGGL((k_pf_attn<D, 4>), gt, dim3(256), 0, s, p);
    };
    if (a.D == 128) go(std::integral_constant<int, 128>{});
    else go(std::integral_constant<int, 64>{});
}
