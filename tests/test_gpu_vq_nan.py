"""The codecs' residual quantisers on samples that are no numbers (csrc/snac.hip: k_vq_level for codebooks of eight dimensions, k_vq_nearest for others and for DAC): codes
stay inside the codebook - the next level reads the table at them -, a latent of NaN takes the first entry as argmax does, other rows of the batch keep their codes."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import dac as odac
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


def _audio(rows, samples):
    audio = (0.3 * np.random.default_rng(samples).standard_normal((rows, samples))).astype(np.float32)
    bad = audio.copy()
    bad[0, samples // 2] = np.nan
    bad[1, 5:9] = [np.inf, -np.inf, np.inf, 3e38]
    return audio, bad


@pytest.mark.parametrize("dim", [8, 5])
def test_snac_codes_of_a_latent_that_is_nan(dim):
    cfg = dict(encoder_dim=6, encoder_rates=[2, 2, 2, 2], decoder_dim=32, decoder_rates=[2, 2, 2, 2], codebook_size=100, codebook_dim=dim, vq_strides=[4, 2, 1])
    dev = mas.SNAC.from_weights(mas.SNACConfig(**cfg), osnac.make_synthetic_weights(osnac.SnacConfig(**cfg), seed=7, with_encoder=True))
    audio, bad = _audio(3, 1000)
    want = dev.encode(audio)
    codes, z = dev.encode(bad, return_latent=True)
    assert np.isnan(z[0]).any() and np.isfinite(z[2]).all()
    for got, ref, stride in zip(codes, want, cfg["vq_strides"]):
        assert got.min() >= 0 and got.max() < cfg["codebook_size"]
        assert np.array_equal(got[2], ref[2])
        lost = np.isnan(z).any(1).reshape(3, -1, stride).any(-1)
        assert lost.any() and (got[lost] == 0).all()


def test_dac_codes_of_a_latent_that_is_nan():
    ocfg = odac.TINY
    W = odac.make_synthetic_weights(ocfg)
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    dev = mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)
    audio, bad = _audio(3, 60 * int(np.prod(ocfg.encoder_rates)))
    want = dev.encode(audio)
    codes, z = dev.encode(bad, return_latent=True)
    assert np.isnan(z[0]).any() and codes.min() >= 0 and codes.max() < ocfg.codebook_size
    assert np.array_equal(codes[2], want[2])
    lost = np.isnan(z).any(1)
    assert (np.moveaxis(codes, 1, -1)[lost] == 0).all()
