"""The three tile shapes of the split-bf16 contraction (csrc/codec_bf3.hip: 128 x 128, 64 x 128, 64 x 64) at their edges: a row gives the same bits alone
(few blocks: the small tiles) and among others (the wide one), and both agree with the oracle."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import dac as odac

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dac():
    # 7 taps of 72 -> 320 and of 160 / 40 channels (dilations 1, 3, 9: both halos), transposed convolutions 320 -> 160 -> 80 -> 40, K of 3 to 23 chunks
    ocfg = odac.DacConfig(encoder_dim=4, encoder_rates=(2, 2), latent_dim=72, decoder_dim=320, decoder_rates=(5, 2, 2), n_codebooks=2, codebook_size=64)
    W = odac.make_synthetic_weights(ocfg)
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    dev = mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)
    return ocfg, odac.DacOracle(ocfg, W), dev


@pytest.mark.parametrize("frames", [1, 13, 25, 26, 63, 64, 65, 129])
def test_tiles_agree(dac, frames):
    ocfg, orc, dev = dac
    codes = np.random.default_rng(frames).integers(0, ocfg.codebook_size, (60, ocfg.n_codebooks, frames)).astype(np.int32)
    many = dev.decode_from_codes(codes)
    ref = orc.decode_from_codes(codes[:1])
    # two planes per operand: 2^-16 of a product and, over a dozen layers, the 3e-4 of tests/test_gpu_dac.py
    assert np.abs(many[:1] - ref).max() <= 3e-4 and np.isfinite(many).all()
    for r in (0, 37):
        assert np.array_equal(dev.decode_from_codes(codes[r:r + 1])[0], many[r])
    assert np.array_equal(dev.decode_from_codes(codes[5:12]), many[5:12])
