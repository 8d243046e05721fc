"""-m gpu: codecs short of memory (codec_run, csrc/codec_kernels.h): where the operands' planes have no room a call goes on without them, with the same bits, in the memory of the f32
tensors and one pre-pass; with less it fails and leaves nothing behind.  The limit is the library's own (mis_debug_device_limit): no allocation reaches the card's."""
import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from mlx_audio_swift_amd import _lib
from mlx_audio_swift_amd.generation import AudioGenerationError
from oracle import dac as odac
from oracle import snac as osnac

pytestmark = pytest.mark.gpu
SNAC = dict(encoder_dim=48, encoder_rates=[2, 4, 8, 8], decoder_dim=1536, decoder_rates=[8, 8, 4, 2], codebook_size=64, codebook_dim=8, vq_strides=[4, 2, 1])


def _held(more=-1):
    return _lib.lib().mis_debug_device_limit(int(more))


def _short(model, call, enough, little):
    """call(model()) with all the memory there is, then with `enough` of what that took, then with `little`: fails, and works again"""
    dev = model()
    before = _held()
    want = call(dev)
    need = _held() - before
    del dev
    for share in enough:
        dev = model()
        _held(share * need)
        try:
            got = call(dev)
            again = call(dev)
        finally:
            _held()
        for g in (got, again, call(dev)):
            assert all(np.array_equal(a, b) for a, b in zip(g, want)), share
        del dev
    dev = model()
    _held(little * need)
    try:
        with pytest.raises(AudioGenerationError):
            call(dev)
    finally:
        _held()
    assert all(np.array_equal(a, b) for a, b in zip(call(dev), want))


def _snac():
    W = osnac.make_synthetic_weights(osnac.SnacConfig(**SNAC), seed=21, with_encoder=True)
    return lambda: mas.SNAC.from_weights(mas.SNACConfig(**SNAC), W)


def test_snac_encode():
    """Three f32 buffers of 48 channels a sample (0.64 of all of it), planes of 96 channels in front of the first strided convolution (1.5 of a buffer, an eighth to spare)."""
    audio = (0.3 * np.random.default_rng(0).standard_normal((2, 200000))).astype(np.float32)

    def call(dev):
        codes, z = dev.encode(audio, return_latent=True)
        return [*codes, z]

    _short(_snac(), call, (0.97, 0.7), 0.5)


def test_snac_decode():
    """Chains of one or two contractions: the second buffer is 3 % of all."""
    ocfg = osnac.SnacConfig(**SNAC)
    codes, noise = osnac.synthetic_codes(ocfg, 2, 24), osnac.synthetic_noise(ocfg, 2, 24)
    _short(_snac(), lambda dev: [dev.decode(codes, noise)], (0.98,), 0.4)


def test_dac_decode():
    ocfg = odac.DacConfig(encoder_dim=4, encoder_rates=(2, 2), n_codebooks=2, codebook_size=64, latent_dim=64, decoder_dim=1536, decoder_rates=(8, 8, 4, 2))
    W = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v
         for k, v in odac.make_synthetic_weights(ocfg).items() if not k.startswith("encoder.")}
    hcfg = mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__})
    codes = np.random.default_rng(1).integers(0, 64, (2, 2, 100)).astype(np.int32)
    _short(lambda: mas.DescriptDAC.from_weights(hcfg, W), lambda dev: [dev.decode_from_codes(codes)], (0.95, 0.85), 0.4)
