"""Causal attention of a prompt pass (csrc/lm_prefill.hip, k_pf_rope_append / k_pf_attn): the edges of its tiles and blocks - 32-key tiles, 32 queries a
wave, 128 or 256 queries a block, 4096-row chunks that cut a row at a position that is no multiple of 32."""
import numpy as np
import pytest

from oracle import llama as ollama

pytestmark = pytest.mark.gpu

WIDE = ollama.LlamaConfig(hidden_size=1024, num_hidden_layers=2, intermediate_size=1024, num_attention_heads=8, num_key_value_heads=1, head_dim=128, vocab_size=640)
# eight kv heads: both shapes below reach 256 blocks of 256 queries, a row alone does not
KV8 = {D: ollama.LlamaConfig(hidden_size=1024, num_hidden_layers=2, intermediate_size=1024, num_attention_heads=16, num_key_value_heads=8, head_dim=D, vocab_size=640)
       for D in (64, 128)}


@pytest.mark.parametrize("ocfg", [ollama.TINY, ollama.TINY_QWEN3, ollama.TINY64, WIDE, KV8[64], KV8[128]], ids=["gqa3", "qknorm", "d64", "gqa8", "wide-d64", "wide-d128"])
@pytest.mark.parametrize("shape", ["edges", "chunks"])
def test_rows_have_the_same_bits_alone_and_in_a_batch_and_match_the_oracle(ocfg, shape):
    """A query's sums run over the key tiles in order whatever block, chunk or batch it belongs to, so a row's logits are the same bits in every
    arrangement.  Against the oracle: the bound of test_gpu_lm.py's logits (max 0.016 of the largest logit)."""
    from gpu_util import logits_errors
    from test_gpu_lm import lm_pair
    W, oracle, dev = lm_pair(ocfg, seed=53)
    rng = np.random.default_rng(3)
    lens = [2, 31, 32, 33, 64, 65, 127, 129, 86, 171, 300] if shape == "edges" else [150] + [100 + b for b in range(40)]      # 41 x 150 > 4096 rows
    rows = [rng.integers(0, ocfg.vocab_size, n).astype(np.int32) for n in lens]
    nxt = rng.integers(0, ocfg.vocab_size, len(rows)).astype(np.int32)
    got = dev.lm_prefill(rows, max_context=320)
    got2 = dev.lm_forward(nxt)
    pick = range(len(rows)) if shape == "edges" else (0, 1, 17, 40)
    for b in pick:
        alone = dev.lm_prefill([rows[b]], max_context=320)
        assert np.array_equal(alone[0], got[b]), lens[b]
        assert np.isfinite(got[b]).all()
    for b in pick:
        oracle.reset(1)
        ref = oracle.forward([np.concatenate([rows[b], nxt[b:b + 1]])], logit_positions=[[lens[b] - 1, lens[b]]])[0].numpy()
        for dv, rf in ((got[b], ref[0]), (got2[b], ref[1])):
            e_max = logits_errors(dv[None], rf[None])[0]
            assert e_max <= 0.016, (lens[b], e_max)
