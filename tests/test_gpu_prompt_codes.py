"""Prompt GEMMs on 8- and 4-bit codes: tiles (csrc/lm_prefill.hip, k_gemm_pf_codes: 64 x 64 with four teams of waves or one, 128 x 128) for more than 64 rows, slices of the
decode step's kernel (csrc/lm_qgemm.hip) for fewer, and for up to 96 of large 4-bit matrices; remainders in rows, columns and groups; ragged prompts.  Against the oracle on the float32 weights
s q + b; and a prompt has the bits that it has alone, whatever kernels its call takes."""
import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from oracle import llama as ollama
from oracle import mlxquant as mq

pytestmark = pytest.mark.gpu


# hidden 1088 = 17 groups, ff 1216 = 19, heads 3 x 128 = 6: quarters of unequal length; 60 and 64 rows: three or more prompts in one slice, 65: the first in tiles; 3072 / 8192 at
# 4 bits: slices of 64 and 16 rows, then tiles; 1024 / 3072: 128 x 128 tiles for gate | up from 641 rows on
@pytest.mark.parametrize("hidden, heads, ff, bits, total", [(1088, 3, 1216, 8, 60), (1088, 3, 1216, 4, 64), (1088, 3, 1216, 8, 64), (1088, 3, 1216, 8, 65), (1088, 3, 1216, 4, 65),
                                                            (3072, 16, 8192, 4, 72), (3072, 16, 8192, 4, 81), (1088, 3, 1216, 8, 75), (1088, 3, 1216, 4, 96), (1088, 3, 1216, 8, 97), (1088, 3, 1216, 4, 431), (1088, 3, 1216, 8, 1000), (1024, 16, 3072, 8, 130),
                                                            (1024, 16, 3072, 4, 333), (1024, 16, 3072, 8, 700), (1024, 16, 4160, 8, 128), (1024, 16, 4160, 4, 129)])
def test_prompts_on_codes(hidden, heads, ff, bits, total):
    from gpu_util import logits_errors
    from gpu_util import lm_host_config
    cfg = ollama.LlamaConfig(hidden_size=hidden, num_hidden_layers=2, intermediate_size=ff, num_attention_heads=heads, num_key_value_heads=1, head_dim=128, vocab_size=640)
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
    rng = np.random.default_rng(total)
    lens, left = [2, 50], total - 52
    while left > 0:
        lens.append(min(left, int(rng.integers(20, 60))))
        left -= lens[-1]
    rows = [rng.integers(0, cfg.vocab_size, n).astype(np.int32) for n in lens]
    many = dev.lm_prefill(rows, max_context=128)
    oracle = ollama.LlamaOracle(cfg, W32, round="bf16")
    for b in range(len(rows)):
        alone = dev.lm_prefill([rows[b]], max_context=128)                                             # one to four tiles of 16 rows
        assert np.array_equal(alone[0], many[b]), (b, lens[b])
    for b in (0, 1, len(rows) - 1):
        oracle.reset(1)
        ref = oracle.forward([rows[b]], logit_positions=[[lens[b] - 1]])[0].numpy()
        e_max, e_rms = logits_errors(many[b][None], ref)[:2]
        assert e_max <= 0.016 and e_rms <= 0.008, (b, e_max, e_rms)                                    # the bounds of test_gpu_loader.py's decode steps
