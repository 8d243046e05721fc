"""-m gpu: the greedy step of the Whisper decoder in one kernel (k_greedy_step) against the launches it stands for (suppress masks, multi-launch sampler, embedding and LayerNorm:
MIS_SAMPLER_WIDE=1): the same ids at vocabularies of part of a pass, several threads' chunks and more than one pass, one, some and more rows than a tile, masks and ranges that cut
the maximum off, rows that end at different steps."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab, d, rows", [(700, 128, 1), (8193, 128, 5), (51866, 384, 3), (57345, 128, 2), (130001, 128, 17)])
def test_greedy_step_has_the_ids_of_the_separate_launches(monkeypatch, vocab, d, rows):
    cfg = mas.WhisperConfig(vocab_size=vocab, num_mel_bins=80, d_model=d, encoder_layers=1, encoder_attention_heads=d // 64, encoder_ffn_dim=256, decoder_layers=1,
                            decoder_attention_heads=d // 64, decoder_ffn_dim=256)
    dev = mas.WhisperModel.synthetic(cfg, seed=vocab)
    rng = np.random.default_rng(vocab)
    wins = [(0.1 * rng.standard_normal(1600 * (i + 1))).astype(np.float32) for i in range(rows)]
    prompt = [vocab - 10, vocab - 9]

    def both(**kw):
        gp = mas.STTGenerateParameters(max_tokens=12, temperature=0.0, **kw)
        one = dev.transcribe_windows(wins, prompt, gp)
        monkeypatch.setenv("MIS_SAMPLER_WIDE", "1")
        want = dev.transcribe_windows(wins, prompt, gp)
        monkeypatch.delenv("MIS_SAMPLER_WIDE")
        assert one == want, kw
        return one

    free = both(eot_id=vocab - 1, timestamp_begin=vocab, suppress_tokens=[], begin_suppress_tokens=[])
    said = sorted({t for r in free for t in r})
    first = [r[0] for r in free if r]
    # what was said is suppressed (twice, with ids outside the vocabulary), then at the first step only, then past the end of the range, then all but one id, then the end of the row
    both(eot_id=vocab - 1, timestamp_begin=vocab, suppress_tokens=said + said + [-1, vocab, vocab + 7], begin_suppress_tokens=first)
    assert all(r[0] not in first for r in both(eot_id=vocab - 1, timestamp_begin=vocab, suppress_tokens=[], begin_suppress_tokens=first) if r)
    both(eot_id=vocab - 1, timestamp_begin=max(said), suppress_tokens=said[:1], begin_suppress_tokens=[])
    both(eot_id=vocab - 1, timestamp_begin=5, suppress_tokens=[0, 1, 3, 4], begin_suppress_tokens=[])
    both(eot_id=free[0][min(3, len(free[0]) - 1)], timestamp_begin=vocab, suppress_tokens=[], begin_suppress_tokens=[])
