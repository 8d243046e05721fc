"""First and last kernel of the codec decoders (codec_embed, k_codec_final): quantisers past a group of four, channels that are no multiple of 4 / 32,
lengths around the 122 outputs of a tile and the 32 frames of an embedding tile."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import dac as odac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_q, dim, latent", [(1, 10, 33), (5, 66, 40), (9, 24, 7)])
def test_tile_edges(n_q, dim, latent):
    ocfg = odac.DacConfig(encoder_dim=4, encoder_rates=(2,), latent_dim=latent, decoder_dim=dim, decoder_rates=(2,), n_codebooks=n_q, codebook_size=16)
    W = odac.make_synthetic_weights(ocfg)
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    dev = mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)
    orc = odac.DacOracle(ocfg, W)
    seen = set()
    for frames in (1, 2, 31, 32, 33, 60, 61, 62, 121, 122, 123):
        codes = np.random.default_rng(frames).integers(-1, ocfg.codebook_size + 1, (2, n_q, frames)).astype(np.int32)
        got = dev.decode_from_codes(codes)
        ref = orc.decode_from_codes(np.clip(codes, 0, ocfg.codebook_size - 1))
        seen.add(got.shape[1] % 122)
        # float32 sums of <= 66 * 7 products through eight layers, |tanh| <= 1: 24 bits times the root of the terms, and the f32 oracle's own
        assert got.shape == ref.shape and np.abs(got - ref).max() <= 2e-5, frames
    assert len(seen) > 6
