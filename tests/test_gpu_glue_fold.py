"""-m gpu: residual + RMSNorm inside the GEMM behind it at one and two rows (`k_gemm_glue`): the bits of the separate launches, at odd and even depth (the residual
stream alternates between two buffers), and of a row among three (separate launches by rule)."""
import numpy as np
import pytest

from oracle import llama as ollama

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 2, 3])
def test_folded_glue_has_the_bits_of_the_separate_launches(monkeypatch, layers):
    from gpu_util import logits_errors
    from test_gpu_lm import lm_pair
    ocfg = ollama.LlamaConfig(hidden_size=3072, num_hidden_layers=layers, intermediate_size=8192, num_attention_heads=24, num_key_value_heads=8, head_dim=128, vocab_size=640)
    W, oracle, dev = lm_pair(ocfg, seed=3)
    toks = np.random.default_rng(5).integers(0, ocfg.vocab_size, (5, 3)).astype(np.int32)
    got = {}
    for rows, fold in ((1, None), (1, "0"), (2, None), (2, "0"), (3, None)):
        monkeypatch.delenv("MIS_GLUE_FOLD", raising=False)
        if fold is not None:
            monkeypatch.setenv("MIS_GLUE_FOLD", fold)
        dev.lm_reset(rows, 64)
        got[rows, fold] = np.stack([dev.lm_forward(t[:rows]) for t in toks])
    assert np.array_equal(got[1, None], got[1, "0"]) and np.array_equal(got[2, None], got[2, "0"])
    assert np.array_equal(got[1, None][:, 0], got[3, None][:, 0]) and np.array_equal(got[2, None], got[3, None][:, :2])
    oracle.reset(1)
    ref = np.stack([oracle.forward([[int(t)]])[0][0].numpy() for t in toks[:, 0]])
    assert logits_errors(got[1, None][:, 0], ref)[0] <= 0.016                                           # the bound of test_gpu_lm.py's logits
