"""-m gpu: Whisper's cross-attention on one (`k_attn_decode<64, 2, true, QP>`), two or four blocks a (row, head) (`k_attn_cross`): a row's logits do
not depend on the split, and every split is within the tolerance that the whole decoder is held to (bf16 at every primitive boundary: 0.022 of the largest logit)."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import whisper as ow

pytestmark = pytest.mark.gpu


def _model(d, heads):
    cfg = ow.WhisperConfig(vocab_size=300, num_mel_bins=80, d_model=d, encoder_layers=1, encoder_attention_heads=heads, encoder_ffn_dim=256, decoder_layers=2,
                           decoder_attention_heads=heads, decoder_ffn_dim=256)
    W = ow.make_synthetic_weights(cfg, seed=d)
    return cfg, ow.WhisperOracle(cfg, W, round="bf16"), mas.WhisperModel.from_weights(mas.WhisperConfig(**{k: getattr(cfg, k) for k in mas.WhisperConfig.__dataclass_fields__}), W)


# (width, heads, rows): four blocks up to 64 (row, head) pairs, two up to 128, one beyond; the projection folded in up to 16 rows (two, three or five
# k-tiles a slice, ragged slices at widths 320 and 832), as slabs beyond
@pytest.mark.parametrize("d,heads,rows,fold", [(256, 4, (1, 16), None), (320, 5, (1, 12, 13, 16), None), (832, 13, (1, 4, 9, 10), None), (640, 10, (1, 6, 7, 13), None),
                                               (256, 4, (1, 16, 17, 32, 33), "0")])
def test_rows_do_not_depend_on_the_split(monkeypatch, d, heads, rows, fold):
    cfg, oracle, dev = _model(d, heads)
    if fold is not None:
        monkeypatch.setenv("MIS_WHISPER_FOLD", fold)
    rng = np.random.default_rng(d)
    feats = (rng.standard_normal((max(rows), 3000, 80)) * 0.5).astype(np.float32)
    toks = rng.integers(0, cfg.vocab_size, (max(rows), 3))
    got = {}
    for B in rows:
        dev.encode(feats[:B])
        dev.decoder_reset()
        got[B] = np.stack([dev.decoder_forward(toks[:B, t]) for t in range(3)], 1)
    for B in rows[1:]:
        assert np.array_equal(got[B][: rows[0]], got[rows[0]]), B
    oracle.reset(2)
    oracle.encode(feats[[0, max(rows) - 1]])
    ref = oracle.decode([toks[0], toks[-1]])
    for i, g in ((0, got[max(rows)][0]), (1, got[max(rows)][-1])):
        r = ref[i].numpy()
        assert np.abs(g - r).max() <= 0.022 * np.abs(r).max()
