"""-m gpu: the SNAC decoder's units of 64 and 128 channels as one kernel each (csrc/codec_x6.hip, k_pw_x6 with taps of 1, 3 and 9): less than a block of 128 columns, part of a second,
a halo longer than what is left of the row, against the oracle - and a row's bits the same alone (chunks of 32 channels) and among others (chunks of 16 from 512 blocks on)."""
import numpy as np
import pytest

from gpu_util import rms, snac_pair
from oracle import snac as osnac

pytestmark = pytest.mark.gpu
CFG = dict(osnac.TINY, vq_strides=[4, 2, 1], codebook_size=64, decoder_dim=1024, decoder_rates=[2, 2, 2, 2], encoder_rates=[2, 2, 2, 2])


@pytest.mark.parametrize("groups", [1, 2, 3, 9])                 # 64, 128, 192, 576 columns of 64 channels, half as many of 128
def test_units_against_the_oracle(groups):
    ocfg, oracle, dev = snac_pair(CFG)
    codes, noise = osnac.synthetic_codes(ocfg, 2, groups), osnac.synthetic_noise(ocfg, 2, groups)
    ref, inter = oracle.decoder(oracle.from_codes(codes), noise, return_intermediates=True)
    got = dev.decode(codes, noise)
    for name in ("block2", "block3"):                            # (the oracle's f32 sums: 2e-5 of the largest value, as behind the transposed convolutions)
        t = dev.debug_tap(name, 2)
        assert t.shape == inter[name].shape and rms(t, inter[name]) < 2e-5 * float(np.abs(inter[name]).max()), name
    assert got.shape == ref.shape and rms(got, ref) < 1e-4


@pytest.mark.parametrize("rows, groups", [(3, 7), (2, 515), (9, 131), (4, 515)])      # 12, 516, 594 and 1032 blocks of 64 channels; a row alone: 4, 258, 66, 258
def test_a_row_alone_has_its_bits(rows, groups):
    ocfg, _, dev = snac_pair(CFG)
    codes, noise = osnac.synthetic_codes(ocfg, rows, groups), osnac.synthetic_noise(ocfg, rows, groups)
    got = dev.decode(codes, noise)
    assert np.isfinite(got).all() and np.abs(got).max() > 0
    assert np.array_equal(dev.decode([c[1:2] for c in codes], [n[1:2] for n in noise])[0], got[1])
