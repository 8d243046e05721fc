// lm_step.h - the layers of a decode step of one or two rows as one launch (lm_step.hip)
#pragma once
#include "lm_kernels.h"

// one weight role: output tiles of 16 columns, K cut into `pieces` of `len` kilobyte tiles - the K ranges of the launch chain's waves (slabs x waves per item),
// whose sums are added in the chain's order
struct StepRole {
    const unsigned char* w;      // layer 0: packed tiles, the K-tiles of a column tile contiguous
    size_t layer;                // bytes from a layer to the next
    int items, K_tiles, pieces, ksb, len;                // items: column tiles, or pairs of gate and up tiles
};
enum { SYNC_TAG = 0, SYNC_LATE = 1, SYNC_WORDS = 32 };
struct StepParams {
    StepRole qkv, o, gu, down;
    const bf16_t *x0, *h0;       // first layer: normalised rows (packed operand), residual stream [Mpad][d]
    bf16_t *x_out, *h_out;       // behind the last layer: model.norm(h) packed, h
    const bf16_t* norms;         // [L][2][d], [d]
    bf16_t *kcache, *vcache;     // [L][rows][Hkv][Smax][D] tiled
    size_t kv_layer;             // elements
    const int* pos;
    const uint8_t* active;
    const float *rope_cos, *rope_sin;
    unsigned char* exch;         // values handed between blocks (step_exch_bytes): cleared, with sync, in front of a request
    unsigned* sync;              // [SYNC_WORDS]: base of the next launch's tags; whether a wait of a step ran out of time
    unsigned* fail;              // sticky: a wait ran out of time (here or in the sampler)
    unsigned long long limit;    // ticks of the 100 MHz counter that a wait may take
    int L, d, H, Hkv, Smax, rows, Mpad;
    int schedule2;               // whose bits attention gives: k_attn_decode2's or (caches past 1024 positions) k_attn_decode's
    float eps, scale;
};
struct StepShape { int L, d, ff, H, Hkv, D, rows; };
size_t step_exch_bytes(const StepShape& s);
// sizes that the launch takes (the device is asked too): otherwise the launch chain
bool step_ok(const StepShape& s, const StepParams& p, int device);
void launch_step(const StepParams& p, hipStream_t s);
// Steps that ran out of time: something that is no call of this process holds compute units (another process, another library's kernels).  The handle's next request stays on the launch
// chain; the next two, four, .. up to 64 if it goes on; a request that gets through ends that.
struct StepPause {
    int skip = 0, next = 1;
    bool due() { return skip == 0 || (--skip, false); }
    void late() { skip = next; next = std::min(2 * next, 64); }
    void fine() { next = 1; }
};
// behind a raised `fail`: whether it was a step's wait, on which `pause` then begins (one line to stderr); the launches have ended
bool step_was_late(const unsigned* sync, StepPause& pause, const char* what);
