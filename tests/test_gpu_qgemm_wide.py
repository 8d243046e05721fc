"""-m gpu: gate and up of quantised checkpoints with 256 blocks of four tiles, at most 16 rows and 33 to 48 scale groups (csrc/lm_qgemm.hip, k_gemm_skinny_q1 of four tiles and eight waves):
waves of four and of five groups, of six, and k_gemm_skinny_q on either side (32 groups; 20 rows).  Decode steps against the oracle on the float32 weights s q + b, and the bits of a row the
same among four others and among nineteen."""
import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from gpu_util import lm_host_config, logits_errors, teacher_forced
from oracle import llama as ollama
from oracle import mlxquant as mq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden, bits", [(2048, 8), (2112, 8), (2304, 4), (3072, 8), (3072, 4)])
def test_gate_and_up_at_few_rows(hidden, bits):
    cfg = ollama.LlamaConfig(hidden_size=hidden, num_hidden_layers=1, intermediate_size=8192, num_attention_heads=2, num_key_value_heads=1, head_dim=128, vocab_size=640)
    dev, W32 = mas.LlamaTTSModel(lm_host_config(cfg)), {}
    for k, v in ollama.make_synthetic_weights(cfg, seed=99).items():
        W32[k] = v
        if v.ndim == 2:
            wq, s, b = mq.quantize(v.float().numpy(), 64, bits)
            s, b = torch.from_numpy(s).bfloat16(), torch.from_numpy(b).bfloat16()
            dev.set_quantized_tensor(k, wq, s, b, 64, bits)
            W32[k] = torch.from_numpy(mq.dequantize(wq, s.float().numpy(), b.float().numpy(), 64, bits))
            if k == "model.embed_tokens.weight":
                W32[k] = W32[k].bfloat16()
        else:
            dev.set_tensor(k, v)
    dev.finalize()
    rng = np.random.default_rng(hidden + bits)
    rows = [rng.integers(0, cfg.vocab_size, 3 + b % 3).astype(np.int32) for b in range(20)]
    oracle = ollama.LlamaOracle(cfg, W32, round="bf16")
    few = teacher_forced(oracle, dev, rows[:5])
    many = teacher_forced(oracle, dev, rows)
    for (l5, ref), (l20, _) in zip(few, many):
        e_max, e_rms, _, agree = logits_errors(l5, ref)
        assert e_max <= 0.016 and e_rms <= 0.008 and agree, (e_max, e_rms)           # the bounds of test_gpu_loader.py's decode steps
        assert np.array_equal(l5, l20)
