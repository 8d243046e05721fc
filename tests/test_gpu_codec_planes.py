"""-m gpu: contractions that hand their output to the next one as bf16 planes (launch_gemm_chain): every width that a decoder has such an edge at, with one column, part of a
tile, whole tiles and a column more, in batches, against the oracle - and a row's bits whatever batch it is in."""
import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from oracle import dac as od

pytestmark = pytest.mark.gpu


def _pair(**kw):
    ocfg = od.DacConfig(encoder_dim=4, encoder_rates=(2, 2), n_codebooks=2, codebook_size=64, **kw)
    W = {k: v for k, v in od.make_synthetic_weights(ocfg).items() if not k.startswith("encoder.")}
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    hcfg = mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__})
    return ocfg, od.DacOracle(ocfg, W), mas.DescriptDAC.from_weights(hcfg, stored)


# 768 -> 384 -> 192 -> 96 channels: three planes in front of the 1x1 of 384, f32 in front of 192 and 96; 1536 -> 768: two planes in front of both; 80 -> 40: no planes
@pytest.mark.parametrize("kw, frames", [
    (dict(latent_dim=64, decoder_dim=768, decoder_rates=(8, 4, 2)), (1, 2, 8, 16, 17)),
    (dict(latent_dim=64, decoder_dim=1536, decoder_rates=(4,)), (1, 16, 32, 33)),
    (dict(latent_dim=40, decoder_dim=80, decoder_rates=(5, 3)), (1, 9)),
], ids=["384-192-96", "768", "40-20"])
def test_planes_between_contractions(kw, frames):
    ocfg, orc, dev = _pair(**kw)
    rng = np.random.default_rng(2)

    def oracle(codes, **kw):
        # (torch's oneDNN transposed convolution is wrong for some of these sizes on some CPUs: two rows of 8 frames, 768 -> 384 channels by 8, differ by 1.7 from each row alone)
        with torch.backends.mkldnn.flags(enabled=False):
            return orc.decode_from_codes(codes, **kw)

    for T in frames:
        codes = rng.integers(0, ocfg.codebook_size, (2, ocfg.n_codebooks, T)).astype(np.int32)
        for bi in range(len(ocfg.decoder_rates)):                          # (a tap wants the block's output in f32, where the decoder goes on from planes alone)
            ref, got = oracle(codes, stop_after=f"block{bi}"), dev.debug_tap(codes, bi)
            assert got.shape == ref.shape and np.abs(got - ref).max() <= 3e-4 * np.abs(ref).max(), (T, bi)
        ref, got = oracle(codes), dev.decode_from_codes(codes)
        assert got.shape == ref.shape and np.abs(got - ref).max() <= 3e-4, T
        np.testing.assert_array_equal(dev.decode_from_codes(codes[1:]), got[1:])


def test_rows_of_columns_that_leave_the_buffers_dirty():
    """The operands' buffers are one per model: a short call behind a long one reads no column of it."""
    ocfg, _, dev = _pair(latent_dim=64, decoder_dim=768, decoder_rates=(8, 4, 2))
    rng = np.random.default_rng(3)
    short, long = (rng.integers(0, ocfg.codebook_size, (b, ocfg.n_codebooks, T)).astype(np.int32) for b, T in ((1, 3), (3, 50)))
    first = dev.decode_from_codes(short)
    dev.decode_from_codes(long)
    np.testing.assert_array_equal(dev.decode_from_codes(short), first)
