"""Rows of many samples in the codecs' f32 contractions (csrc/codec_f32.hip): 2^22 samples are 175 s at 24 kHz; from 2^24 on the offsets inside a tile no
longer fit 32 bits.  A row's first samples are the same bits as a short row's (the decoder looks a few frames ahead, not further)."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


# last block: 5 channels (rows and channels that end inside a tile), and 80 (two row tiles)
@pytest.mark.parametrize("dim, groups", [(80, 258), (80, 1030), (1280, 1030)], ids=["past-4M", "past-16M", "past-16M-two-row-tiles"])
def test_decode(dim, groups):
    cfg = dict(encoder_dim=6, encoder_rates=[8, 8, 8, 8], decoder_dim=dim, decoder_rates=[8, 8, 8, 8], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    ocfg = osnac.SnacConfig(**cfg)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), osnac.make_synthetic_weights(ocfg, seed=4))
    dev.set_noise(False, seed=3)                                   # NoiseBlocks with noise: the contraction under test runs on whole rows
    codes = osnac.synthetic_codes(ocfg, 1, groups)
    got = dev.decode(codes)[0, 0]
    assert got.size == groups * 4 * 4096 and np.isfinite(got).all() and np.abs(got[-4096:]).max() > 0
    short = dev.decode([c[:, :c.shape[1] // groups * 12] for c in codes])[0, 0]
    keep = short.size - 16 * 4096                                  # 3 frames of the stem, 39 / 8 of the first block's units, less of the others see the end
    assert np.array_equal(got[:keep], short[:keep])
