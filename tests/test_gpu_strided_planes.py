"""The SNAC encoder's strided convolutions on three planes of the phase split (k_enc_phase_planes, csrc/codec_bf3.hip): as accurate as the f32 kernels, the bits of a row whatever its
call - quarters of K in blocks of their own or one after the other, 64 x 64 or 64 x 128 tiles - and values past the largest bfloat16."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from gpu_util import codec_exact_f32
from oracle import snac as osnac

pytestmark = pytest.mark.gpu

CFG = dict(encoder_dim=48, encoder_rates=[2, 4, 8, 8], decoder_dim=64, decoder_rates=[8, 8, 4, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])


# one frame of codes (a column behind the last stride) alone, in eight rows and, twelve columns, in 48; a row whose K = 3072 has 456 blocks of 64 x 128; a call in which a tile takes its quarters itself
@pytest.mark.parametrize("rows, samples", [(1, 2048), (8, 2048), (48, 6000), (1, 60001), (1, 151111), (48, 24000)])
def test_strided_convolutions(rows, samples):
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**CFG), seed=21, with_encoder=True)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**CFG), W)
    oracle = osnac.SnacOracle(osnac.SnacConfig(**CFG), W, dtype=np.float64)
    audio = (0.3 * np.random.default_rng(samples).standard_normal((rows, samples))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    with codec_exact_f32():
        _, z32 = dev.encode(audio[:1], return_latent=True)
    ref = oracle.encoder(oracle.preprocess(audio[:1, None].astype(np.float64)))
    err, err32 = (np.sqrt(np.mean((g[:1] - ref) ** 2) / np.mean(ref ** 2)) for g in (z, z32))
    assert err <= 1.25 * err32 and err32 <= 1e-5, (err, err32)             # (f32 sums in another order: see test_gpu_codec_split3.py)
    one, z1 = dev.encode(audio[rows - 1:], return_latent=True)
    assert np.array_equal(z1[0], z[rows - 1]) and all(np.array_equal(a[0], c[rows - 1]) for a, c in zip(one, codes))


# scale 1e-30: the channel is all that the last convolution gives, nothing but a depthwise convolution behind it; 1e-36 in front of other blocks: a share of order ten, for which sine
# is not the other kernel's to the last bits (the lower planes of such weights are subnormal) - no infinity and no NaN
@pytest.mark.parametrize("block, scale", [(1, 1e-36), (2, 1e-36), (3, 1e-36), (4, 1e-30)])
def test_values_past_the_largest_bfloat16(block, scale):
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**CFG), seed=22, with_encoder=True)
    p = "encoder.block.layers.%d.block.layers." % block
    W[p + "2.block.layers.3.bias"][5] = 3.4e38                             # the last unit's channel 5, through a Snake that is none
    W[p + "3.alpha"][0, 5] = 0.0
    W[p + "4.weight_v"][:, :, 5] *= scale
    dev = mas.SNAC.from_weights(mas.SNACConfig(**CFG), W)
    audio = (0.3 * np.random.default_rng(4).standard_normal((1, 30001))).astype(np.float32)
    _, z = dev.encode(audio, return_latent=True)
    with codec_exact_f32():
        _, z32 = dev.encode(audio, return_latent=True)
    assert np.isfinite(z32).all() and np.isfinite(z).all()
    if block == 4:
        assert np.abs(z).max() > 1e4 and np.abs(z - z32).max() <= 1e-5 * np.abs(z32).max()
