"""The many-rows form of the prompt GEMMs (csrc/lm_prefill.hip, k_gemm_pf_wide over gemm_tiles.h): tiles of 128, 160 and 192 rows, remainders in rows and
columns, several tiles a block, K of exactly the ring's three k-steps; packed rows of ragged prompts.  A row has the bits it has alone (k_gemm_pf_ring)."""
import numpy as np
import pytest

from oracle import llama as ollama

pytestmark = pytest.mark.gpu


# rows in all: 2500 .. 4090 of the largest chunk; N = 640 / 1088 / 2432 (not whole 256-column tiles), K = 192 (three k-steps), 384, 1088, 1216: the 128 x 128 tiles where K is
# short and their blocks few, the others here.  2112 wide: every product here, on 128 rows a tile (1333), 160 (3333) and 192 (4090)
@pytest.mark.parametrize("hidden, heads, ff, total", [(1088, 3, 1216, 2500), (1088, 3, 1216, 3333), (1088, 3, 1216, 4090), (192, 8, 1216, 4075), (2112, 16, 1216, 1333),
                                                      (2112, 16, 1216, 3333), (2112, 16, 1216, 4090)])
def test_rows_of_ragged_prompts_have_the_bits_they_have_alone(hidden, heads, ff, total):
    from gpu_util import logits_errors
    from test_gpu_lm import lm_pair
    ocfg = ollama.LlamaConfig(hidden_size=hidden, num_hidden_layers=2, intermediate_size=ff, num_attention_heads=heads, num_key_value_heads=1, head_dim=128, vocab_size=640)
    W, oracle, dev = lm_pair(ocfg, seed=11)
    rng = np.random.default_rng(total)
    lens, left = [2, 1, 129, 3], total - 135
    while left > 0:
        lens.append(min(left, int(rng.integers(100, 150))))
        left -= lens[-1]
    rows = [rng.integers(0, ocfg.vocab_size, n).astype(np.int32) for n in lens]
    many = dev.lm_prefill(rows, max_context=160)
    for b in (0, 2, 3, len(rows) - 1):                                                                 # (one token alone takes the decode step)
        assert np.array_equal(dev.lm_prefill([rows[b]], max_context=160)[0], many[b]), lens[b]
    oracle.reset(1)
    ref = oracle.forward([rows[2]], logit_positions=[[lens[2] - 1]])[0].numpy()
    assert logits_errors(many[2][None], ref)[0] <= 0.016                                              # the bound of test_gpu_lm.py's logits
