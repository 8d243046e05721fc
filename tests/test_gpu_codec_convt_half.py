"""-m gpu: the transposed convolutions of stride 2 in blocks of 62 columns (k_x6_convt_half, few blocks): a row alone, which takes them, against the same row in a batch of so many that the
blocks of 126 columns do it - the same bits, with and without the NoiseBlock, one and two tiles of rows, one and four chunks of channels, columns around a block's edge."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


# channels in -> out of the last block: 64 -> 32, 128 -> 64; columns in front of it: 4 x 4 a group and one less (62 and 126 lie between 3 and 4, 7 and 8 groups)
@pytest.mark.parametrize("noise", [True, False])
@pytest.mark.parametrize("dim", [128, 256])
@pytest.mark.parametrize("groups", [1, 3, 4, 5, 7, 8, 16])
def test_a_row_alone_and_among_others(dim, noise, groups):
    ocfg = osnac.SnacConfig(**dict(osnac.TINY, decoder_rates=[4, 2], decoder_dim=dim, vq_strides=[4, 2, 1], noise=noise))
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), osnac.make_synthetic_weights(ocfg))
    rows = 300
    rng = np.random.default_rng(groups)
    codes = [rng.integers(0, ocfg.codebook_size, (rows, groups * k)).astype(np.int32) for k in (1, 2, 4)]
    many = dev.decode(codes)
    alone = dev.decode([c[:1] for c in codes])
    assert np.array_equal(alone[0], many[0]) and np.isfinite(alone).all() and np.abs(alone).max() > 0
