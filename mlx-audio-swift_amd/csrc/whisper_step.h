// whisper_step.h - all decoder layers of a Whisper step as one launch (whisper_step.hip)
#pragma once
#include "lm_kernels.h"
#include "lm_step.h"

#include <vector>

enum { WS_QKV, WS_O, WS_CQ, WS_CO, WS_FC1, WS_FC2, WS_ROLES };
// one entry per layer, and one behind the last whose first norm is the decoder's
struct WsLayer { const bf16_t *w[WS_ROLES], *b[WS_ROLES], *lnw[3], *lnb[3]; };
// column tiles of 16, K cut as the launch chain cuts it (slabs, then the waves of an item); `per` tiles a block, blocks [first, first + blocks)
struct WsRole { int tiles, KT, S, ksb, per, first, blocks; };
// what a block has for all layers: one matrix or attention; tiles of every matrix, or both attentions of a (row, head)
enum { WS_ALL, WS_SHARED };
struct WsParams {
    WsRole role[WS_ROLES];
    int what;
    int self_first, cross_first, blocks;                                  // a block per (row, head)
    const WsLayer* layers;
    const unsigned* table;       // ws_tables
    const bf16_t *x0, *h0;       // first layer: normalised rows (packed operand), residual stream [Mpad][d]
    bf16_t* x_out;               // behind the last layer: LayerNorm(h), packed
    bf16_t *self_k, *self_v, *cross_k, *cross_v;
    size_t self_layer, cross_layer;                                       // elements
    const int* pos;
    const uint8_t* active;
    unsigned char* exch;         // values handed between blocks (ws_exch_bytes): cleared, with sync, in front of a request
    unsigned *sync, *fail;                                                // as StepParams'
    unsigned long long limit;
    int L, d, ff, H, rows, Smax, Spad, cross_len, units, k_max;
    float eps, scale;
};
size_t ws_exch_bytes(const WsParams& p);
// fills the blocks' roles; false: sizes that stay on the launch chain
bool ws_plan(WsParams& p, int device);
// who multiplies what: the pieces of a block's tiles dealt to its waves
std::vector<unsigned> ws_tables(const WsParams& p);
void launch_whisper_step(const WsParams& p, hipStream_t s);
