"""The four-wave encoder GEMMs (csrc/whisper_kernels.hip, k_gemm_rows over gemm_tiles.h): tiles of 128, 160, 192 and 256 rows, remainders in rows and columns,
several tiles a block, every epilogue, cache tiles with swapped operands.  The bits of the 128 x 128 kernel and k_scatter_kv (`MIS_GEMM_BIG3=0`)."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas

pytestmark = pytest.mark.gpu


# 1280 wide: the largest model's shapes (q|k|v and cross k|v on 128, 160, 192 and 256 rows by the number of windows); 640: columns that are no whole tiles, plain
# q|k|v with its own scatter; 576 with K = 576 = nine k-steps
@pytest.mark.parametrize("d, heads, ff, rows", [(1280, 20, 5120, n) for n in (2, 3, 4, 6, 8)] + [(640, 10, 1088, 8), (640, 10, 2560, 11), (576, 9, 1728, 13)])
def test_encoder_gemms_have_the_bits_of_the_small_tiles(monkeypatch, d, heads, ff, rows):
    cfg = mas.WhisperConfig(vocab_size=700, num_mel_bins=128, d_model=d, encoder_layers=1, encoder_attention_heads=heads, encoder_ffn_dim=ff, decoder_layers=1,
                            decoder_attention_heads=heads, decoder_ffn_dim=ff)
    dev = mas.WhisperModel.synthetic(cfg, seed=rows)
    feats = np.random.default_rng(rows).standard_normal((rows, 3000, 128)).astype(np.float32)
    got = {}
    for big in ("0", "1"):
        monkeypatch.setenv("MIS_GEMM_BIG3", big)
        got[big] = dev.encode(feats)
        dev.decoder_reset()
        got[big + "d"] = dev.decoder_forward([7] * rows)                                              # the cross keys and values
    monkeypatch.delenv("MIS_GEMM_BIG3")
    assert np.isfinite(got["0"]).all() and np.abs(got["0"]).max() > 0
    assert np.array_equal(got["0"], got["1"]) and np.array_equal(got["0d"], got["1d"])
