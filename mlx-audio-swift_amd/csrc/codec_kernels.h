// codec_kernels.h - f32 kernels shared by the codec back ends (SNAC decoder, Soprano / Vocos decoder); defined in snac.hip
#pragma once
#include "common.h"
#include <vector>

enum { GEMM_PLAIN = 0, GEMM_RESID = 1, GEMM_NOISE = 2, GEMM_CONVT = 3, GEMM_GELU = 4, GEMM_TAPS = 5 };

// Snake, x + sin^2(alpha x) ra, with the factor as `a` = alpha / pi (snake_alpha below, rounded once when the weights are laid out): f = a x less its nearest
// whole number, rounded once (fmaf: the rounding of the product alone, kept in the difference, is 1.15 times the error from |alpha x| = ten on), and sin^2(pi f),
// |f| <= 1/2, is f^2 times a polynomial of degree five in f^2 (least maximum, found by reweighted least squares; 5.9e-9 before rounding).  Eleven VALU instructions:
// the product alpha x reduced by multiples of pi and the square of a polynomial for the sine were fourteen, in kernels that then issued VALU in 60 - 90 % of their cycles (50 - 80 now).
// Off 64 bits by 4.5e-8 (rms) where |alpha x| is about one, 1.01e-7 at three, 3.15e-7 at ten, 3.11e-6 at a hundred: rounding of a.  The form before: 5.1e-8, 1.08e-7,
// 3.15e-7, 3.10e-6.
__device__ __forceinline__ float mis_snake(float x, float a, float ra) {
    const float f = fmaf(a, x, -rintf(a * x));
    const float s = f * f;
    float p = fmaf(s, -3.27294594e+0f, 1.29907303e+1f);
    p = fmaf(s, p, -3.00859532e+1f);
    p = fmaf(s, p, 4.27253848e+1f);
    p = fmaf(s, p, -3.24695811e+1f);
    p = fmaf(s, p, 9.86960292e+0f);
    return fmaf(ra, p * s, x);
}
inline float snake_alpha(float alpha) { return (float)((double)alpha * 0.31830988618379067154); }

// z[c][t] = sum over q in order of tables[q][code(q, t)][c]: a block takes 32 channels x 32 frames (table rows are read along c, z written along t); four
// quantisers' codes, then their table rows are requested together (one by one they were two dependent round trips per quantiser and frame: SNAC
// 10.5 -> 5.1 us for 48 frames, DAC 26 -> 7 us for 250 frames of twelve quantisers)
template <class Code>
__device__ __forceinline__ void codec_embed(const float* __restrict__ tables, int n_q, int bins, int C, int T, float* __restrict__ z, Code code) {
    __shared__ float tile[32][33];
    const int c0 = blockIdx.y * 32, t0 = blockIdx.x * 32, cc = threadIdx.x & 31, r0 = threadIdx.x >> 5, c = min(c0 + cc, C - 1);
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int q0 = 0; q0 < n_q; q0 += 4) {
        int id[4][4];
        float v[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) id[q][r] = code(min(q0 + q, n_q - 1), min(t0 + r0 + 8 * r, T - 1));
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[q][r] = tables[((size_t)min(q0 + q, n_q - 1) * bins + min(max(id[q][r], 0), bins - 1)) * C + c];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = q0 + q < n_q ? acc[r] + v[q][r] : acc[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) tile[cc][r0 + 8 * r] = acc[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int co = c0 + r0 + 8 * r, t = t0 + cc;
        if (co < C && t < T) z[(size_t)co * T + t] = tile[r0 + 8 * r][cc];
    }
}

// NoiseBlock noise (MLXRandom.normal([B,1,T]), Layers.swift:274): Box-Muller on mis-synth-v1 uniforms keyed by (seed, block, GLOBAL row, t)
__device__ __forceinline__ float codec_noise_value(uint64_t key, uint64_t row, int n) {
    const uint64_t u = mis_splitmix64((key ^ (row * 0xD1B54A32D192ED03ull)) + (uint64_t)n);
    const float u1 = ((float)(uint32_t)(u >> 40) + 0.5f) * 5.9604644775390625e-08f;
    const float u2 = ((float)(uint32_t)((u >> 16) & 0xFFFFFF) + 0.5f) * 5.9604644775390625e-08f;
    return sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
}

// Per-model state of the split-bf16 path (codec_bf3.hip): packed hi/lo weight fragments keyed by the A^T pointer (packed on first use,
// on the calling stream) and the split-activation scratch planes.  One in-flight call per model handle, as for the rest of the engine.
struct CodecPack {
    struct Entry { const float* at; int ntaps, Cin, M, Cp, KS, MT32; uint16_t* wp; };
    std::vector<Entry> entries;
    struct X6 { const float* at; int ntaps, Cin, M, KS, MT32; uint16_t* wp; };
    std::vector<X6> x6;   // three-plane fragments (codec_x6.hip)
    DevBuf<uint16_t> planes[2];          // operands: written by the epilogue in front (in turns), or split by a pre-pass into the one that this call's epilogue does not write
    bool plain = false;                  // no epilogue writes planes (codec_run)
    DevBuf<float> part;   // split-K slabs of launch-shaped contractions (GemmParams.split_k_ok)
    CodecPack() {}
    CodecPack(const CodecPack&) = delete;
    CodecPack& operator=(const CodecPack&) = delete;
    ~CodecPack();
    const Entry& get(const float* at, int ntaps, int Cin, int M, hipStream_t s);
    const X6& get_x6(const float* at, int ntaps, int Cin, int M, hipStream_t s);
};

// One call of a codec.  Where it runs out of memory, the planes are given back and it runs once more without them - the pre-pass alone, half of the memory; the same bits
template <class F> void codec_run(CodecPack& pack, F body) {
    try { body(); return; }
    catch (const MisNoMemory&) { if (!pack.planes[0].p && !pack.planes[1].p) throw; }
    for (auto& b : pack.planes) b.release();                          // (waits for the device)
    struct Plain { bool& on; explicit Plain(bool& b) : on(b) { on = true; } ~Plain() { on = false; } } plain(pack.plain);
    body();
}

// Decoders open a scope around their launches: launch_gemm picks the scope's CodecPack up when GemmParams.pack is null.  Encoders (codebook decisions) open
// one with bf3 = false: the three-plane contractions, which are as accurate as the f32 kernels, and none of two planes.  null: exact-f32 kernels only.
struct CodecPackScope {
    CodecPack *prev, *prev_x6;
    explicit CodecPackScope(CodecPack* p, bool bf3 = true);
    ~CodecPackScope();
};
CodecPack* codec_x6_scope();          // the innermost scope's, or null
bool codec_exact_f32();               // MIS_CODEC_EXACT_F32=1

// (strided convolutions: their input's, two taps)
struct CodecPlanes;
bool codec_planes_strided(const struct GemmParams& p, int batch, CodecPlanes& out);
// An operand as bf16 planes, time-major: [n planes, stride elements apart][batch][Tp][Cp]; row r holds column r + t_org, through Snake where alpha is given.
// ends: rows without a column are zero (an operand of one tap does not need them)
struct CodecPlanes {
    uint16_t* p;
    int n, Cp, Tp, t_org;
    bool ends;
    size_t stride;
    const float *alpha, *ralpha;
};
// A wave's 32 x 32 C/D tile (column lane & 31, row (r & 3) + 8 (r >> 2) + 4 (lane >> 5)) to NP bf16 planes, each the nearest to what is left, through CP_LDS(NP) bytes of LDS of its
// own: put takes registers 0 - 7 (r0 = 0) and 8 - 15 (r0 = 8) - lanes l and l + 32 trade halves, so that each writes eight consecutive channels - and flush stores 64 bytes of a
// column's channels per four lanes (straight from the registers they were 32.  96 x 96 with residual, 80043 columns: 28 us without planes, 42 and 36 with; the pre-pass 15).
// Three planes: a value past the largest bfloat16 has that one as its first.
// (one plane of eight values, two to a word; v: what is left)
__device__ __forceinline__ void codec_split_pairs(float (&v)[8], uint32_t (&w)[4], bool clamp) {
    constexpr float TOP = 3.38953138925153547590470800371487866880e+38f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float &a = v[2 * i], &b = v[2 * i + 1];
        const float ca = clamp ? __builtin_amdgcn_fmed3f(a, -TOP, TOP) : a, cb = clamp ? __builtin_amdgcn_fmed3f(b, -TOP, TOP) : b;
        w[i] = (uint32_t)f32_to_bf16(ca) | ((uint32_t)f32_to_bf16(cb) << 16);
        a -= __uint_as_float(w[i] << 16);
        b -= __uint_as_float(w[i] & 0xffff0000u);
    }
}
// (registers 0 - 7 or 8 - 15 of a 32 x 32 C/D tile: lanes l and l + 32 trade halves, then each holds eight consecutive channels of its column - an MFMA-B fragment of 16 channels)
__device__ __forceinline__ uint4 codec_tile_piece(float (&y)[8], bool clamp) {
    uint32_t w[4];
    codec_split_pairs(y, w, clamp);
    const auto s0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false), s1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    return make_uint4(s0[0], s1[0], s0[1], s1[1]);
}
#define CP_LD 40
#define CP_LDS(NP) ((NP) * 32 * CP_LD)       // in bf16
template <int NP>
__device__ __forceinline__ void codec_tile_put(float (&y)[8], uint16_t* st, int r0, int lane) {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        *reinterpret_cast<uint4*>(st + (q * 32 + (lane & 31)) * CP_LD + 2 * r0 + 8 * (lane >> 5)) = codec_tile_piece(y, NP == 3 && q == 0);
    }
}
// d: channel 0 of the tile in row 0; row(c): the operand's row of the tile's column c, < 0: none
template <int NP, class Row>
__device__ __forceinline__ void codec_tile_flush(const uint16_t* st, uint16_t* d, size_t stride, int Cp, int lane, Row row) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = i * 16 + (lane >> 2), r = row(c);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint4 v = *reinterpret_cast<const uint4*>(st + (q * 32 + c) * CP_LD + (lane & 3) * 8);
            if (r >= 0) *reinterpret_cast<uint4*>(d + q * stride + (size_t)r * Cp + (lane & 3) * 8) = v;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// rows without a column, [0, -t_org) and behind column T, of the channels [c0, c0 + nc): by the blocks that hold the first and the last columns
__device__ __forceinline__ void codec_plane_ends(const CodecPlanes& o, int b, int T, int c0, int nc, bool first, bool last, int tid, int threads) {
    if (!o.ends) return;
    const int lo = max(0, -o.t_org), hi = min(o.Tp, T - o.t_org), i0 = first ? 0 : lo, rows = lo + (last ? o.Tp - hi : 0) - i0, per = nc / 8 * o.n;
    for (int i = tid; i < rows * per; i += threads) {
        const int r = i0 + i / per, j = i % per;
        *reinterpret_cast<uint4*>(o.p + (size_t)(j / (nc / 8)) * o.stride + ((size_t)b * o.Tp + (r < lo ? r : hi + r - lo)) * o.Cp + c0 + j % (nc / 8) * 8) = make_uint4(0, 0, 0, 0);
    }
}

#define CODEC_DW_HALO 27              // 3 * max dilation (9)
struct PwFusedParams {
    const float* X; const float* R; float* Y;
    const float *w7, *b1, *a1, *ra1;       // DW: depthwise weights [C][7], bias, Snake before the taps
    const float *a2, *ra2;                 // Snake in front of the 1x1 conv
    const float *AT, *b2;                  // W2^T [C][C] ([k][m]), bias
    int T, dil, ldx, ldr, ldy;
    int nbx, per, tiles;                   // blocks of columns a row, blocks an XCD, blocks (the launcher's)
    const CodecPlanes* out;                // units without taps: the operand of the contraction behind, or null
};
// three-plane split of the unit tails (codec_x6.hip); false: no pack, exact-f32 asked for, or another width - nothing launched
bool launch_pw_x6(int C, bool dw, const PwFusedParams& p, CodecPack* pack, int batch, hipStream_t s);

struct GemmParams {
    CodecPack* pack;      // non-null: MFMA-bound shapes run as split-bf16 contractions (codec_bf3.hip); null: exact-f32 kernels only
    const float* AT;      // [K][M]   (CONVT: [s][K][M], K = 2*Cin)
    const float* bias;    // [M] or null
    const float* X;       // [B][Kx][Tin]  (Kx = K; CONVT: Cin)
    float* Y;             // [B][M][Tout]
    const float* R;       // RESID, TAPS (or null): [B][M][N]
    const float* scale;   // with R: optional per-row scale of (acc + bias)  (ConvNeXt gamma)
    const float* noise;   // NOISE: explicit [B][N], or null
    int noise_rng;        // NOISE with noise == null: 1 = draw N(0,1) from the documented generator, 0 = zeros
    uint64_t noise_key;   // (seed, block) key of the generator
    const int32_t* row_ids;   // optional global row id per batch row (rng keyed by GLOBAL row)
    int64_t row_offset;
    const float* alpha;   // Snake prologue on X rows (null = none): alpha / pi (snake_alpha), here and wherever a kernel takes a Snake
    const float* ralpha;
    int M, K, N;          // N = output columns per phase
    int Tin, Tout;
    int s, pad, Cin;      // CONVT only (Cin also TAPS)
    int ldx, ldy;         // row strides of X and of Y / R in floats; 0 = dense (Tin, Tout)
    int x_lo;             // lowest valid X column (<= 0): columns [x_lo, 0) hold carried history (streaming decode), zero below
    int dup_bias_n0;      // CONVT: add the bias a second time to output frame n = 0 - the reference's streaming overlap-add sums
                          // two biased outputs there (DecoderBlockUpsample.step, Qwen3TTSSpeechTokenizer.swift:553-576)
    int split_k_ok;       // 1x1 modes on the split-bf16 path: the launch may split its K range over blocks when one batch row gives too few
                          // blocks to fill the chip (the factor depends on the SHAPE only, never on the batch: a row's result is the same
                          // whatever batch it shares); float32 slabs summed in slice order by a second launch that applies the epilogue
    int taps, dil;        // TAPS: dense conv, K = taps*Cin, tap j reads x[:, n - pad + j*dil] (zero outside); A^T row j*Cin + c;
                          // pad = (taps-1)*dil: causal, (taps-1)*dil/2: "same"; optional R (+scale) residual epilogue
};
// snake: Snake prologue on the X rows (CONVT always runs it: pass alpha = ralpha = zeros for identity)
// out: the operand of the contraction behind; true: written (and p.Y with it if keep), false: p.Y as ever
bool launch_gemm(int mode, bool snake, const GemmParams& p, int batch, hipStream_t s, const CodecPlanes* out = nullptr, bool keep = true);
// exact-f32 kernels (codec_f32.hip): every mode but CONVT, TAPS without Snake; p must have ldx / ldy resolved
void launch_gemm_f32(int mode, bool snake, const GemmParams& p, int batch, hipStream_t s);
// k-tap contractions of K >= 1024 add four partial sums, over the ranges [codec_quarter(w), codec_quarter(w + 1)) of their steps of 16 channels of a tap, in order:
// in waves that run beside each other or one after the other - the same bits, whatever the length and the batch
bool codec_quarters(const GemmParams& p);
__host__ __device__ inline int codec_quarter(int steps, int w) { return w >= 4 ? steps : steps * w / 16 * 4; }
// three-plane split (codec_x6.hip): 1x1 and k-tap contractions of at least 48 rows and a multiple of 16 channels; false: not eligible, nothing launched
bool launch_gemm_x6(int mode, bool snake, const GemmParams& p, int batch, hipStream_t s, const CodecPlanes* out = nullptr);
// (out: whether the forms of codec_x6.hip write it: two planes, of as many channels as they have rows)
inline bool codec_x6_writes_planes(int mode, const GemmParams& p, const CodecPlanes& out) { return mode == GEMM_RESID && p.M % 32 == 0 && out.n == 2 && out.Cp == p.M; }
// three-plane split: transposed convolution of stride 2, two taps per phase, 32 .. 64 rows, behind Snake; false: another shape
// noise: with the NoiseBlock behind it (its X is p.Y, its Y unused)
bool launch_convt_x6(const GemmParams& p, int batch, hipStream_t s, const GemmParams* noise = nullptr);
// split-bf16 path; false = shape not eligible (or MIS_CODEC_EXACT_F32=1), nothing launched.  p must have ldx / ldy resolved
// in: the operand is there already (codec_planes of the same call); out: the epilogue also writes (p.Y null: only) the operand of the contraction behind
bool launch_gemm_bf3(int mode, bool snake, const GemmParams& p, int batch, hipStream_t s, const CodecPlanes* in = nullptr, const CodecPlanes* out = nullptr);
bool bf3_writes_planes(int mode, const GemmParams& p);
bool bf3_takes_convt(const GemmParams& p);
// the operand of this call as the epilogue in front of it can write it (scope's pack, buffer `slot`); false: the call wants f32
bool codec_planes(int mode, bool snake, const GemmParams& p, int batch, int slot, CodecPlanes& out);
// depthwise 7-tap conv (zero padded, dilation dil): shorter odd kernels ride in centred 7-tap weights
void launch_dw7(const float* X, float* Y, const float* w7 /*[C][7]*/, const float* bias, int batch, int C, int T, int dil, hipStream_t s);
// Snake -> 7-tap conv (C -> 1, weights at w[c cs + k ks]) -> tanh
void launch_codec_final(const float* X, float* out, int64_t out_stride, const float* w, int cs, int ks, float bias, const float* alpha, const float* ralpha, int batch, int C, int T,
                        hipStream_t s);
// encoder pieces (SNAC / DAC): first conv k7 "same" 1 -> C (w [C][7]); Snake + phase split for a stride-s conv of kernel 2 s
// and padding p = ceil(s / 2) (y[(c*s + r)][m] = snake(x[c][s*m + r - p]), m <= T / s); nearest code of the L2-normalised latent (first index on ties; cn = normalised codebook
// [CB][CD], cn2 = its squared norms); residual -= table[code] (table [CB][C], code index t / stride)
void launch_enc_first(const float* audio, float* y, const float* w, const float* bias, int batch, int C, int T, hipStream_t s);
void launch_enc_phase_split(const float* x, float* y, const float* a, const float* ra, int batch, int C, int T, int stride, hipStream_t s);
void launch_vq_nearest(const float* ze, const float* cn, const float* cn2, int32_t* codes, int batch, int CD, int CB, int Tm, hipStream_t s);
void launch_vq_residual(float* r, const int32_t* codes, const float* table, int batch, int C, int T, int stride, hipStream_t s);

// Contractions one behind the other, each reading the output of the one in front (g.X = its g.Y): where both sides can, that output goes over as the planes its reader
// multiplies, and as f32 only if something else reads it (keep)
struct CodecOp { int mode; bool snake, keep; GemmParams g; };
void launch_gemm_chain(const CodecOp* ops, int n, int batch, hipStream_t s);
