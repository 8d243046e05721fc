"""The residual quantiser of SNAC's encoder (csrc/snac.hip: k_vq_level, one launch a level, for codebooks of eight dimensions; four kernels for others) from the
latent the encoder returns: channels and entries that are no whole block, strides of 1 to 6, one level, several rows."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim, enc, entries, strides, rows, samples", [(8, 6, 100, [4, 2, 1], 3, 1000), (8, 48, 4096, [4, 2, 1], 1, 4096), (8, 20, 257, [1], 2, 700),
                                                                       (8, 24, 300, [6, 3, 2, 1], 5, 333), (5, 6, 100, [4, 2, 1], 2, 1000)])
def test_codes_are_the_nearest_entries(dim, enc, entries, strides, rows, samples):
    cfg = dict(encoder_dim=enc, encoder_rates=[2, 2, 2, 2], decoder_dim=32, decoder_rates=[2, 2, 2, 2], codebook_size=entries, codebook_dim=dim, vq_strides=strides)
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**cfg), seed=7, with_encoder=True)
    dev, oracle = mas.SNAC.from_weights(mas.SNACConfig(**cfg), W), osnac.SnacOracle(osnac.SnacConfig(**cfg), W, dtype=np.float64)
    audio = (0.3 * np.random.default_rng(rows).standard_normal((rows, samples))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    alone = dev.encode(audio)                                             # without the latent: the same codes
    ref, dist = oracle.quantize(z.astype(np.float64), return_details=True)
    open_row = np.ones(rows, bool)                                        # a tie taken the other way changes the levels behind it
    for got, again, want, d in zip(codes, alone, ref, dist):
        assert np.array_equal(got, again) and got.min() >= 0 and got.max() < entries
        s = np.sort(d, -1)
        sure = (s[..., 1] - s[..., 0]) > 1e-5                             # distances of unit vectors in f32: 1e-6
        assert np.array_equal(got[open_row][sure[open_row]], want[open_row][sure[open_row]])
        open_row &= (got == want).all(-1)
    assert open_row.mean() > 0.5


# From 1537 codes of a level on a block owns four neighbours (the last block of a row fewer): the codes that a row has alone, one code a block
@pytest.mark.parametrize("strides, rows, samples", [([4, 2, 1], 17, 1617), ([1], 3, 9511), ([6, 3, 2, 1], 29, 1137)])
def test_codes_do_not_depend_on_the_codes_of_a_block(strides, rows, samples):
    cfg = dict(encoder_dim=24, encoder_rates=[2, 2, 2, 2], decoder_dim=32, decoder_rates=[2, 2, 2, 2], codebook_size=700, codebook_dim=8, vq_strides=strides)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**cfg), osnac.make_synthetic_weights(osnac.SnacConfig(**cfg), seed=5, with_encoder=True))
    audio = (0.3 * np.random.default_rng(rows).standard_normal((rows, samples))).astype(np.float32)
    many, z = dev.encode(audio, return_latent=True)
    assert many[-1].size > 1536
    for b in range(rows):
        alone, za = dev.encode(audio[b:b + 1], return_latent=True)
        assert np.array_equal(za[0], z[b]) and all(np.array_equal(a[0], m[b]) for a, m in zip(alone, many)), b
