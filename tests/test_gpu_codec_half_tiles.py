"""Which tile the split-bf16 contractions of two and seven taps take among many blocks (csrc/codec_bf3.hip): 128 x 128 for whole row tiles (256 and 128 rows), 64 x 128 with
two blocks a compute unit for others (192, 96, 48).  The bits of the small tiles of a few blocks, and the oracle's values."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import dac as odac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [512, 384])
@pytest.mark.parametrize("frames", [33, 129])
def test_tiles_of_many_blocks(dim, frames):
    ocfg = odac.DacConfig(encoder_dim=4, encoder_rates=(2, 2), latent_dim=64, decoder_dim=dim, decoder_rates=(5, 2, 2), n_codebooks=2, codebook_size=64)
    W = odac.make_synthetic_weights(ocfg)
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    dev = mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)
    codes = np.random.default_rng(frames).integers(0, ocfg.codebook_size, (60, ocfg.n_codebooks, frames)).astype(np.int32)
    many = dev.decode_from_codes(codes)
    ref = odac.DacOracle(ocfg, W).decode_from_codes(codes[:1])
    # two planes per operand: 2^-16 of a product and, over a dozen layers, the 3e-4 of tests/test_gpu_dac.py
    assert np.abs(many[:1] - ref).max() <= 3e-4 and np.isfinite(many).all()
    for r in (0, 37):
        assert np.array_equal(dev.decode_from_codes(codes[r:r + 1])[0], many[r])
