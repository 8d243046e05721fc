"""The three-plane contractions (csrc/codec_x6.hip) - the fused residual units: both column tiles and chunk depths, 96 / 128 / 192 channels; the 1x1 and k-tap form: one to
eight row tiles per block; column and row remainders in both - as accurate as the exact-f32 kernels, and the same bits whatever batch (and with it tile or
chunk depth) a row comes in."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from gpu_util import codec_exact_f32
from oracle import dac as odac
from oracle import encodec as oencodec
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_bf3(monkeypatch):
    """The two-plane contractions off: what is left of the error is the f32 kernels' and the three-plane kernel's."""
    monkeypatch.setenv("MIS_BF3_MIN_K", "1000000")
    monkeypatch.setenv("MIS_BF3_MIN_K1", "1000000")


def check(dev, orc, codes, rows, pick):
    """rows of codes as one batch; the first two against the oracle (SNAC: 64 bits, DAC: float32)."""
    ref = orc(pick(codes, slice(0, 2)))
    got = dev(codes)
    with codec_exact_f32():
        f32 = dev(codes)
    err, err32 = (np.sqrt(np.mean((g[:2] - ref) ** 2) / np.mean(ref ** 2)) for g in (got, f32))
    assert not np.array_equal(got, f32)                    # the other kernel did run
    # both are float32 sums in another order: the same size within the scatter of a few thousand samples, and under 24-bit sums through ten layers
    assert err <= 1.25 * err32 and err32 <= 1e-5, (err, err32)
    for r in (0, rows - 1):
        assert np.array_equal(dev(pick(codes, slice(r, r + 1)))[0], got[r])


# decoder channels 128 (units), 256 and 128 (NoiseBlock); 384, 192, 96, 48 (1x1 residuals, and rows past a tile of 32)
@pytest.mark.parametrize("dim", [256, 512, 768])
@pytest.mark.parametrize("rows, groups", [(3, 5), (20, 60), (40, 60)], ids=["one-wave", "two-waves", "many"])
def test_snac(no_bf3, dim, rows, groups):
    cfg = dict(encoder_dim=8, encoder_rates=[2, 2, 2, 8], decoder_dim=dim, decoder_rates=[8, 2, 2, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    ocfg = osnac.SnacConfig(**cfg)
    W = osnac.make_synthetic_weights(ocfg, seed=31, with_encoder=True)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), W)
    dev.set_noise(True)
    oracle = osnac.SnacOracle(ocfg, W, dtype=np.float64)
    codes = osnac.synthetic_codes(ocfg, rows, groups)
    check(dev.decode, lambda c: oracle.decode(c, None), codes, rows, lambda c, sl: [x[sl] for x in c])


@pytest.mark.parametrize("rows, frames", [(2, 9), (9, 211)], ids=["one-wave", "many"])
def test_dac_192_96(no_bf3, rows, frames):
    ocfg = odac.DacConfig(encoder_dim=4, encoder_rates=(2, 2), latent_dim=40, decoder_dim=384, decoder_rates=(8, 5, 2), n_codebooks=2, codebook_size=64)
    W = odac.make_synthetic_weights(ocfg)
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    dev = mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)
    orc = odac.DacOracle(ocfg, W)
    codes = np.random.default_rng(3).integers(0, ocfg.codebook_size, (rows, ocfg.n_codebooks, frames)).astype(np.int32)
    check(dev.decode_from_codes, orc.decode_from_codes, codes, rows, lambda c, sl: c[sl])


# encoder channels 48 .. 768: strided convolutions of two taps over 2 - 8 phases of 48 - 384 channels, one short row to many
@pytest.mark.parametrize("rows, samples", [(1, 4096 + 31), (12, 9 * 4096 - 5)], ids=["short", "many"])
def test_snac_encode(rows, samples):
    cfg = dict(encoder_dim=48, encoder_rates=[2, 2, 2, 8], decoder_dim=32, decoder_rates=[8, 2, 2, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    ocfg = osnac.SnacConfig(**cfg)
    W = osnac.make_synthetic_weights(ocfg, seed=12, with_encoder=True)
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), W)
    oracle = osnac.SnacOracle(ocfg, W, dtype=np.float64)
    audio = (0.3 * np.random.default_rng(8).standard_normal((rows, samples))).astype(np.float32)
    codes, z = dev.encode(audio, return_latent=True)
    with codec_exact_f32():
        _, z32 = dev.encode(audio, return_latent=True)
    ref = oracle.encoder(oracle.preprocess(audio[:1, None].astype(np.float64)))
    err, err32 = (np.sqrt(np.mean((g[:1] - ref) ** 2) / np.mean(ref ** 2)) for g in (z, z32))
    assert not np.array_equal(z, z32) and err <= 1.25 * err32 and err32 <= 1e-5, (err, err32)
    one, z1 = dev.encode(audio[rows - 1:], return_latent=True)
    assert np.array_equal(z1[0], z[rows - 1]) and all(np.array_equal(a[0], c[rows - 1]) for a, c in zip(one, codes))


# one channel of one frame's code is infinite, or finite past the largest bfloat16 (3.39e38): the 1x1 behind the first depthwise convolution gives what
# the f32 kernel gives - infinities of the same sign, finite sums of finite products
@pytest.mark.parametrize("gain", [1e30, 3.4e8], ids=["infinite", "past-bf16"])
@pytest.mark.parametrize("rows", [1, 40, 160, 300], ids=["narrow", "two-tiles", "four-tiles", "eight-tiles"])
def test_values_that_three_planes_do_not_hold(gain, rows):
    cfg = dict(encoder_dim=8, encoder_rates=[2, 2, 2, 8], decoder_dim=512, decoder_rates=[8, 2, 2, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])
    ocfg = osnac.SnacConfig(**cfg)
    W = dict(osnac.make_synthetic_weights(ocfg, seed=31))
    q = [k for k in W if "quantizers.0" in k or "quantizers.layers.0" in k]
    book, g, v = (next(k for k in q if k.endswith(e)) for e in ("codebook.weight", "out_proj.weight_g", "out_proj.weight_v"))
    W[book] = np.array(W[book])
    W[book][:, 0] = W[book][5] = 0.0
    W[book][5, 0] = 1e30                                           # code 5: (1e30, 0, ...), and out_proj takes it to channel 17 alone
    W[g], W[v] = np.array(W[g]) * 0 + 1e-30, np.array(W[v]) * 0
    W[v].reshape(W[v].shape[0], -1)[:, 1] = 1.0
    W[v].reshape(W[v].shape[0], -1)[17] = np.eye(8)[0]
    W[g].reshape(-1)[17] = gain
    sg, sv = (next(k for k in W if "decoder.model.layers.0" in k and k.endswith(e)) for e in ("weight_g", "weight_v"))
    W[sv] = np.zeros_like(W[sv])
    W[sv].reshape(W[sv].shape[0], -1)[:, slice(0, 7) if gain == 1e30 else 3] = 1.0      # (0 times infinity would be NaN; 7 times 3.4e38 infinite)
    W[sg] = np.ones_like(W[sg])
    dev = mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), W)
    dev.set_noise(True)
    codes = [np.where(c == 5, 6, c).astype(np.int32) for c in osnac.synthetic_codes(ocfg, rows, 9)]
    codes[0][:, 3] = 5
    dev.decode(codes)
    got = dev.debug_tap("stem_pw", rows)
    with codec_exact_f32():
        f32 = dev.debug_tap("stem_pw", rows)
    hit = np.abs(f32) > 1e30
    assert hit.any() and not hit.all() and np.isinf(f32[hit]).all() == (gain == 1e30) and not np.isnan(f32).any()
    if gain == 1e30:
        assert np.array_equal(got[hit], f32[hit])
    else:
        assert np.abs(got[hit] / f32[hit] - 1).max() <= 1e-6       # one product is larger than all others by 1e38
    assert np.abs(got[~hit] - f32[~hit]).max() <= 1e-5 * np.abs(f32[~hit]).max()


@pytest.mark.parametrize("value", [np.inf, 3.4e38], ids=["infinite", "past-bf16"])
def test_encodec_with_a_channel_that_three_planes_do_not_hold(value):
    """The LSTM's input projection (1x1) saturates its gates, and the transposed convolution of stride 2 (identity in front) stays finite where f32 does."""
    ocfg = oencodec.EncodecConfig(num_filters=32, codebook_size=64, codebook_dim=32, hidden_size=32, upsampling_ratios=(2, 2), target_bandwidths=(8.0,), sampling_rate=1600)
    W = {k: np.array(v) for k, v in oencodec.make_synthetic_weights(ocfg).items()}
    W["decoder.layers.0.conv.bias"][17] = value
    dev = mas.Encodec.from_weights(mas.EncodecConfig(**{k: getattr(ocfg, k) for k in mas.EncodecConfig.__dataclass_fields__ if hasattr(ocfg, k)}), W)
    codes = np.random.default_rng(0).integers(0, ocfg.codebook_size, (2, ocfg.num_quantizers, 9)).astype(np.int32)
    for stage in (2, 3):
        got = dev.debug_tap(codes, stage)
        with codec_exact_f32():
            f32 = dev.debug_tap(codes, stage)
        fin = np.isfinite(f32)
        assert np.array_equal(got[~fin], f32[~fin], equal_nan=True) and np.isfinite(got[fin]).all(), stage
        # the first convolution runs on two planes there and in f32 here (1e-5); relative to the largest of the channel
        g, f = np.where(fin, got, 0), np.where(fin, f32, 0)
        assert np.all(np.abs(g - f) <= 1e-4 * np.maximum(np.abs(f).max(axis=2, keepdims=True), 1e-3)), stage
        assert fin.sum() >= f32.size * 127 // 128 or (stage == 3 and value == np.inf)      # (the identity is a Snake of rate 0: 0 times infinity)
