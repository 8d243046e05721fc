"""Copies of more than 4 MB between device memory and pageable memory go through a pinned ring with several threads (HostRing, csrc/host_util.cpp):
sizes that end inside a chunk, more chunks than slots, both directions - the same bits as rows small enough for the plain copy."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac
from oracle import whisper as owhisper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,groups", [(5, 103), (9, 257)])                 # 4.2 MB: 3 chunks; 18.9 MB: 10 chunks in 8 slots
def test_out(rows, groups):
    ocfg = osnac.SnacConfig(**{**osnac.TINY, "decoder_rates": [8, 8, 4, 2]})
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), osnac.make_synthetic_weights(ocfg, seed=3))
    dev.set_noise(True)
    codes = osnac.synthetic_codes(ocfg, rows, groups)
    got = dev.decode(codes)
    assert got.nbytes > (4 << 20) and got.nbytes % (2 << 20)
    for r in range(rows):
        one = dev.decode([c[r:r + 1] for c in codes])
        assert one.nbytes < (4 << 20) and np.array_equal(one[0], got[r])


def test_in_and_out():
    ocfg = owhisper.TINY
    W = owhisper.make_synthetic_weights(ocfg, seed=5)
    dev = mas.WhisperModel.from_weights(mas.WhisperConfig(**{k: getattr(ocfg, k) for k in ocfg.__dataclass_fields__}), W)
    rng = np.random.default_rng(1)
    feats = rng.standard_normal((11, 3000, ocfg.num_mel_bins)).astype(np.float32)
    got = dev.encode(feats)                                                    # 10.6 MB in, 8.4 MB out
    for b in (0, 5, 10):
        assert np.array_equal(dev.encode(feats[b:b + 1])[0], got[b])
