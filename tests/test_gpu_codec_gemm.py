"""The exact-f32 contractions of the codecs (csrc/codec_f32.hip) where their tiles end: row and column remainders of the 32 / 64 / 128 tiles, channels that are
no multiple of 4 or 16, the encoders' k-split form, and a batch that picks another tile than its rows alone (same bits)."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from oracle import snac as osnac

pytestmark = pytest.mark.gpu

# decoder channels 40, 20, 10, 5 (no multiples of 16, then of 4); encoder channels 6 .. 96
ODD = dict(encoder_dim=6, encoder_rates=[2, 2, 2, 2], decoder_dim=80, decoder_rates=[4, 2, 2, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
# decoder channels 512 .. 64: the wide tiles once 24 rows of 9 frames come together, the small tile for one row; encoder convolutions with K >= 1024
WIDE = dict(encoder_dim=32, encoder_rates=[2, 2, 4, 8], decoder_dim=1024, decoder_rates=[8, 2, 2, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])


def pair(cfg):
    ocfg = osnac.SnacConfig(**cfg)
    W = osnac.make_synthetic_weights(ocfg, seed=77, with_encoder=True)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), W)
    dev.set_noise(True)
    return ocfg, osnac.SnacOracle(ocfg, W, dtype=np.float64), dev


@pytest.mark.parametrize("cfg", [ODD, WIDE], ids=["odd", "wide"])
@pytest.mark.parametrize("groups", [1, 9])
def test_decode(cfg, groups):
    ocfg, oracle, dev = pair(cfg)
    rows = 24
    codes = osnac.synthetic_codes(ocfg, rows, groups)
    got = dev.decode(codes)
    ref = oracle.decode([c[:2] for c in codes], None)
    # float32 sums (<= 1e-6 per layer) and the split-bf16 products of the wide layers (1e-5): the waveform gate of test_gpu_snac.py is 1e-4
    assert np.sqrt(np.mean((got[:2] - ref) ** 2)) <= 1e-4 * max(1e-3, np.sqrt(np.mean(ref ** 2)))
    for r in (0, 23):
        assert np.array_equal(dev.decode([c[r:r + 1] for c in codes])[0], got[r])


@pytest.mark.parametrize("cfg", [ODD, WIDE], ids=["odd", "wide"])
@pytest.mark.parametrize("samples", [257, 4096 + 31])
def test_encode(cfg, samples):
    ocfg, oracle, dev = pair(cfg)
    rng = np.random.default_rng(5)
    audio = (0.3 * rng.standard_normal((5, samples))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    ref = oracle.encoder(oracle.preprocess(audio[:2, None].astype(np.float64)))
    assert np.sqrt(np.mean((z[:2] - ref) ** 2)) <= 1e-5 * np.sqrt(np.mean(ref ** 2))          # float32 sums over K <= 3072 through nine layers
    one, z1 = dev.encode(audio[3:4], return_latent=True)
    assert np.array_equal(z1[0], z[3]) and all(np.array_equal(a[0], c[3]) for a, c in zip(one, codes))


# the same with a first convolution of 64 rows over K >= 1024
LONG_K = dict(WIDE, encoder_rates=[16, 2, 2, 2])


@pytest.mark.parametrize("exact", [False, True], ids=["three-planes", "f32"])
@pytest.mark.parametrize("cfg", [WIDE, LONG_K], ids=["wide", "long-k"])
def test_a_recording_and_its_beginning_have_the_same_bits(cfg, exact, monkeypatch):
    """The strided convolutions' sums are taken in an order that only the matrix decides: the frames of a long recording that do not see where the short one
    ends have its bits, on either side of the lengths - and batches - where the kernels' forms take turns."""
    if exact:
        monkeypatch.setenv("MIS_CODEC_EXACT_F32", "1")
    ocfg, oracle, dev = pair(cfg)
    audio = (0.3 * np.random.default_rng(9).standard_normal((1, 1400 * 128))).astype(np.float32)
    _, z = dev.encode(audio, return_latent=True)
    for frames in (80, 300, 700):
        _, short = dev.encode(audio[:, :frames * 128], return_latent=True)
        assert np.array_equal(short[:, :, :frames - 48], z[:, :, :frames - 48]), frames
    _, many = dev.encode(np.repeat(audio, 10, axis=0), return_latent=True)
    assert np.array_equal(many[0], z[0]) and np.array_equal(many[9], z[0])
