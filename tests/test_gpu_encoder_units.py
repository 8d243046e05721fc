"""The SNAC encoder's units of 48 and 96 channels as one kernel each (csrc/codec_x6.hip, k_pw_x6 with taps) where 512 blocks of 128 columns run: the bits of the
depthwise kernel and the 1x1 contraction (`MIS_CODEC_FUSED_UNITS=0`) at the line, at columns that are no whole block, over several rows."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


# strides of 2 and 8: 48 channels at 65536 (512 blocks), 67584 and 150 x 512 samples, 96 channels at half of them
@pytest.mark.parametrize("rows, samples", [(1, 65536), (1, 70001), (150, 500), (3, 50001)])
def test_fused_units_have_the_bits_of_two_kernels(monkeypatch, rows, samples):
    cfg = dict(encoder_dim=48, encoder_rates=[2, 4, 8, 8], decoder_dim=64, decoder_rates=[8, 8, 4, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**cfg), seed=rows, with_encoder=True)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**cfg), W)
    audio = (0.3 * np.random.default_rng(rows).standard_normal((rows, samples))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    monkeypatch.setenv("MIS_CODEC_FUSED_UNITS", "0")
    codes2, z2 = dev.encode(audio, return_latent=True)
    assert np.isfinite(z).all() and np.abs(z).max() > 0
    assert np.array_equal(z, z2) and all(np.array_equal(a, b) for a, b in zip(codes, codes2))


# Values past the largest bfloat16 behind a Snake that is none (alpha 0): their planes are infinite, the sums of the two kernels' contractions no numbers, and both take
# them again in f32 - the same bits, finite, in a row of many blocks as in one of few
@pytest.mark.parametrize("block", [1, 2])
def test_sums_past_the_planes_are_those_of_two_kernels(monkeypatch, block):
    cfg = dict(encoder_dim=48, encoder_rates=[2, 4, 8, 8], decoder_dim=64, decoder_rates=[8, 8, 4, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**cfg), seed=3, with_encoder=True)
    unit = "encoder.block.layers.%d.block.layers.2.block.layers." % block
    W[unit + "2.alpha"][0, 5] = 0.0
    W[unit + "1.bias"][5] = 3.4e38
    W[unit + "3.weight_v"][:, 0, 5] *= 1e-36
    dev = mas.SNAC.from_weights(mas.SNACConfig(**cfg), W)
    audio = (0.3 * np.random.default_rng(9).standard_normal((1, 131073))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    monkeypatch.setenv("MIS_CODEC_FUSED_UNITS", "0")
    codes2, z2 = dev.encode(audio, return_latent=True)
    assert np.isfinite(z2).all() and np.array_equal(z, z2) and all(np.array_equal(a, b) for a, b in zip(codes, codes2))
