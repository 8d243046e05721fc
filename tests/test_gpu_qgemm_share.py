"""-m gpu: a scale group's share of a sum in the kernels of four n-tiles a wave (csrc/lm_qgemm.hip, qg_share): which of its two products is rounded is part of a decode step's bits.
Codes of one power of two q and bias = -q scale: the products are each other's negatives, so a group gives what the rounding of one of them left, with the sign of the other -
fma(bias, sum x, scale * sum q x) in all groups of a wave but its last one or two, fma(scale, sum q x, bias * sum x) there.  x = +-w, chosen so that its sums are exact."""
import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from gpu_util import lm_host_config
from oracle import llama as ollama

pytestmark = pytest.mark.gpu


def _model(d, ff, vocab, coded, wide_norm, bits, rng, top):
    """Embeddings of +-1, attention that adds nothing, `wide_norm`'s weights 8 bits times 2^(top - 11 .. top); coded: name -> scales, biases [rows][groups]"""
    cfg = ollama.LlamaConfig(hidden_size=d, num_hidden_layers=1, intermediate_size=ff, num_attention_heads=1, num_key_value_heads=1, head_dim=128, vocab_size=vocab, tie_word_embeddings=False)
    W = {k: torch.zeros(s, dtype=torch.bfloat16) for k, s in (
        ("model.embed_tokens.weight", (vocab, d)), ("model.norm.weight", (d,)), ("lm_head.weight", (vocab, d)), ("model.layers.0.input_layernorm.weight", (d,)),
        ("model.layers.0.post_attention_layernorm.weight", (d,)), ("model.layers.0.self_attn.q_proj.weight", (128, d)), ("model.layers.0.self_attn.k_proj.weight", (128, d)),
        ("model.layers.0.self_attn.v_proj.weight", (128, d)), ("model.layers.0.self_attn.o_proj.weight", (d, 128)), ("model.layers.0.mlp.gate_proj.weight", (ff, d)),
        ("model.layers.0.mlp.up_proj.weight", (ff, d)), ("model.layers.0.mlp.down_proj.weight", (d, ff)))}
    emb = rng.choice([-1.0, 1.0], (32, d)).astype(np.float32)
    W["model.embed_tokens.weight"][:32] = torch.from_numpy(emb).bfloat16()
    w = (rng.integers(128, 256, d) / 128.0 * 2.0 ** (top - rng.integers(0, 12, d))).astype(np.float32)
    W["model.norm.weight"] += 1.0
    W[wide_norm] = torch.from_numpy(w).bfloat16()
    sums = (emb * w).astype(np.float64).reshape(32, -1, 64).sum(-1)                  # [token][group], exact in f32
    assert np.array_equal(sums, sums.astype(np.float32))
    coded = coded(sums)
    dev = mas.LlamaTTSModel(lm_host_config(cfg))
    for k, v in W.items():
        if k in coded:
            s, b = coded[k]
            n, q = s.shape[0], {8: 0x80808080, 4: 0x88888888}[bits]
            dev.set_quantized_tensor(k, np.full((n, d * bits // 32), q, np.uint32), torch.from_numpy(s).bfloat16(), torch.from_numpy(b).bfloat16(), 64, bits)
        else:
            if k == "model.layers.0.mlp.down_proj.weight" and "pick" in coded:
                v[torch.arange(d), torch.from_numpy(coded["pick"])] = 1.0
            if k == "lm_head.weight" and "pick" in coded:
                v[torch.arange(d), torch.arange(d)] = 1.0
            dev.set_tensor(k, v)
    dev.finalize()
    return dev, emb, sums


def _left(scale, q, sums, waves):
    """what a group alone gives to every row: [token][row], group row % groups"""
    G = sums.shape[1]
    first = np.zeros(G, bool)
    for i in range(waves):
        a, b = G * i // waves, G * (i + 1) // waves
        first[a:a + max(b - a - 1, 0) // 2 * 2] = True
    g = np.arange(len(scale)) % G
    v = q * scale.astype(np.float64)[None] * sums[:, g]                              # exact: 8 + 24 bits
    return np.where(first[g], -1.0, 1.0) * (v - v.astype(np.float32)), first[g]


def _alone(scale, q, G):
    s, b = np.zeros((2, len(scale), G), np.float32)
    rows = np.arange(len(scale))
    s[rows, rows % G] = scale
    b[rows, rows % G] = -q * scale
    return s, b


# waves of two, four and five groups; 5 rows and 20: one and two tiles of rows
@pytest.mark.parametrize("d, bits", [(512, 8), (1088, 8), (1088, 4)])
def test_output_projection(d, bits):
    rng, V, q = np.random.default_rng(d + bits), 65536, {8: 128.0, 4: 8.0}[bits]
    scale = (rng.integers(128, 256, V) / 128.0).astype(np.float32)
    dev, _, sums = _model(d, 256, V, lambda sums: {"lm_head.weight": _alone(scale, q, d // 64)}, "model.norm.weight", bits, rng, 0)
    left, first = _left(scale, q, sums, 4)
    for rows in (5, 20):
        dev.lm_reset(rows, 16)
        got = dev.lm_forward(np.arange(rows, dtype=np.int32))
        assert np.array_equal(got, left[:rows].astype(np.float32)), rows              # (at most 8 bits: nothing left to round)
    assert all((left[:, m] != 0).mean() > 0.3 for m in (first, ~first) if m.any())


# 33 groups over eight waves: four and five; 48: six each.  5 rows k_gemm_skinny_q1, 20 rows k_gemm_skinny_q; 2048: k_gemm_skinny_q at both
@pytest.mark.parametrize("d, bits", [(2048, 8), (2112, 8), (3072, 8), (3072, 4)])
def test_gate_and_up(d, bits):
    rng, ff, q, G = np.random.default_rng(d + bits), 8192, {8: 128.0, 4: 8.0}[bits], d // 64
    scale = (rng.integers(128, 256, ff) / 128.0).astype(np.float32)
    pick = rng.permutation(ff)[:d]
    P = "model.layers.0.mlp."

    def coded(sums):
        gs, gb = np.zeros((2, ff, G), np.float32)                                     # gate: 64 or so for one token, whatever the others make of it
        gb[:, 0] = 64.0 / np.abs(sums[:, 0]).max()
        return {P + "gate_proj.weight": (gs, gb), P + "up_proj.weight": _alone(scale, q, G), "pick": pick}

    dev, emb, sums = _model(d, ff, max(d, 512), coded, P.replace("mlp.", "post_attention_layernorm.weight"), bits, rng, 10 if bits == 8 else 14)
    left, first = _left(scale, q, sums, 8)
    bf = lambda a: torch.from_numpy(np.asarray(a, np.float32)).bfloat16().double().numpy()
    gate = bf(bf(64.0 / np.abs(sums[:, 0]).max()) * sums[:, :1])
    act = bf(bf(gate * bf(1.0 / (1.0 + np.exp(-gate)))) * bf(left))
    h = bf(emb + act[:, pick])
    want = h / np.sqrt((h * h).mean(-1, keepdims=True) + 1e-5)
    other = bf(emb - act[:, pick])
    for rows in (5, 20):
        dev.lm_reset(rows, 16)
        got = dev.lm_forward(np.arange(rows, dtype=np.int32))[:, :d]
        err = np.abs(got - want[:rows]) - 0.012 * np.abs(want[:rows])                 # three roundings to bf16 (2^-9 each) and the sums of the norm
        assert (err <= 0).all(), (rows, err.max(), (err > 0).mean())
    far = np.abs(other - h) > 0.1 * np.abs(h)                                             # (outputs that the other form would put elsewhere)
    assert all(far[:5][:, first[pick] == m].mean() > 0.1 for m in (True, False))
