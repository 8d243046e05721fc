"""The few-rows form of the prompt GEMMs (csrc/lm_prefill.hip, k_gemm_pf_ring): row remainders of its 32-row tiles, K of fewer k-steps than its ring and more;
the bits of the 128 x 128 tiles, which a row meets in a large batch."""
import numpy as np
import pytest

from oracle import llama as ollama

pytestmark = pytest.mark.gpu


# K = 256 / 512 (4 and 8 k-steps: inside the ring) and 1536 / 2560 (24 and 40)
@pytest.mark.parametrize("hidden, ff", [(256, 512), (1536, 2560)])
def test_short_prompts_have_the_bits_of_the_large_batch(hidden, ff):
    from gpu_util import logits_errors
    from test_gpu_lm import lm_pair
    ocfg = ollama.LlamaConfig(hidden_size=hidden, num_hidden_layers=2, intermediate_size=ff, num_attention_heads=hidden // 128, num_key_value_heads=1, head_dim=128,
                              vocab_size=640)
    W, oracle, dev = lm_pair(ocfg, seed=5)
    rng = np.random.default_rng(7)
    lens = [2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 97] + [120] * 49                                   # 60 rows of 120: the large tiles for all but hidden 256
    rows = [rng.integers(0, ocfg.vocab_size, n).astype(np.int32) for n in lens]
    many = dev.lm_prefill(rows, max_context=128)
    for b in range(11):
        alone = dev.lm_prefill([rows[b]], max_context=128)[0]
        few = dev.lm_prefill(rows[max(0, b - 1):b + 1], max_context=128)[-1]
        assert np.array_equal(alone, many[b]) and np.array_equal(few, many[b]), lens[b]
    oracle.reset(1)
    ref = oracle.forward([rows[10]], logit_positions=[[96]])[0].numpy()
    assert logits_errors(many[10][None], ref)[0] <= 0.016                                             # the bound of test_gpu_lm.py's logits
