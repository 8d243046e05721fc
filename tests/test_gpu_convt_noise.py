"""-m gpu: the last transposed convolutions of a SNAC decoder with the NoiseBlock behind them in one kernel (k_x6_convt, 64 and 32 rows): part of a block of 126 columns, a block
and a few columns, many, against the oracle - and a row's bits whatever batch it is in."""
import numpy as np
import pytest

from gpu_util import rms, snac_pair
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 4, 8, 33])               # 16, 64, 128, 528 columns of 64 rows, twice as many of 32
def test_noise_behind_the_transposed_convolution(groups):
    ocfg, oracle, dev = snac_pair(dict(osnac.TINY, vq_strides=[4, 2, 1], codebook_size=64, decoder_dim=512, decoder_rates=[2, 2, 2, 2], encoder_rates=[2, 2, 2, 2]))
    codes, noise = osnac.synthetic_codes(ocfg, 2, groups), osnac.synthetic_noise(ocfg, 2, groups)
    ref, inter = oracle.decoder(oracle.from_codes(codes), noise, return_intermediates=True)
    got = dev.decode(codes, noise)
    for name in ("block2", "block3"):
        t = dev.debug_tap(name, 2)
        assert t.shape == inter[name].shape and rms(t, inter[name]) < 2e-5 * float(np.abs(inter[name]).max()), name
    assert got.shape == ref.shape and rms(got, ref) < 1e-4
    assert np.array_equal(dev.decode([c[1:] for c in codes], [n[1:] for n in noise])[0], got[1])
