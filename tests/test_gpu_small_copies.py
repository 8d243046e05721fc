"""-m gpu: codes, samples and latents that go between the device and the caller's memory by a kernel through pinned memory (csrc/host_util.cpp, HostRing) against the same call on device
memory, which takes plain copies: odd lengths (no multiple of 16 bytes), the edge of what is small (1 MiB together, 64 KiB of codes) and past it."""
import ctypes as C

import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from mlx_audio_swift_amd import _lib
from oracle import dac as od
from oracle import snac as osnac

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def snac():
    ocfg = osnac.SnacConfig(encoder_dim=16, decoder_dim=64)
    return mas.SNAC.from_weights(mas.SNACConfig(**{k: getattr(ocfg, k) for k in mas.SNACConfig.__dataclass_fields__}), osnac.make_synthetic_weights(ocfg, with_encoder=True))


@pytest.fixture(scope="module")
def dac():
    ocfg = od.DacConfig(latent_dim=40, decoder_dim=80, encoder_dim=4, encoder_rates=(2, 2), decoder_rates=(8, 5, 4, 2))
    W = {k: v for k, v in od.make_synthetic_weights(ocfg).items() if not k.startswith("encoder.")}
    stored = {k.replace(".outProj.", ".out_proj.").replace(".inProj.", ".in_proj.").replace("decoder.model.", "decoder.model.layers."): v for k, v in W.items()}
    return mas.DescriptDAC.from_weights(mas.DescriptDACConfig(**{k: getattr(ocfg, k) for k in mas.DescriptDACConfig.__dataclass_fields__}), stored)


# 2048 samples a group: 128 groups are 1 MiB of samples; 8, 3 x 100: past it; 2341 groups of one row: past 64 KiB of codes
@pytest.mark.parametrize("rows,groups", [(1, 1), (1, 12), (3, 7), (1, 128), (2, 64), (1, 129), (3, 100), (1, 2400)])
def test_snac_decode(snac, rows, groups):
    rng = np.random.default_rng(rows * 1000 + groups)
    codes = [rng.integers(0, 4096, (rows, groups * k)).astype(np.int32) for k in (1, 2, 4)]
    host = snac.decode(codes)
    on = [torch.from_numpy(c).cuda() for c in codes]
    out = torch.zeros(host.shape, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ptr = (C.c_void_p * 3)(*[c.data_ptr() for c in on])
    assert _lib.lib().mis_snac_decode(snac._h, ptr, rows, groups, None, out.data_ptr()) == 0
    assert np.array_equal(host, out.cpu().numpy()) and np.abs(host).max() > 0


@pytest.mark.parametrize("rows,samples", [(1, 1), (1, 12001), (3, 30011), (2, 151111), (4, 240000)])
def test_snac_encode(snac, rows, samples):
    rng = np.random.default_rng(samples)
    a = (0.1 * rng.standard_normal((rows, samples))).astype(np.float32)
    codes, z = snac.encode(a, return_latent=True)
    on = torch.from_numpy(a).cuda()
    out = [torch.zeros(c.shape, dtype=torch.int32, device="cuda") for c in codes]
    zo = torch.zeros(z.shape, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ptr = (C.c_void_p * len(out))(*[o.data_ptr() for o in out])
    assert _lib.lib().mis_snac_encode(snac._h, on.data_ptr(), rows, samples, ptr, zo.data_ptr()) == 0
    assert all(np.array_equal(c, o.cpu().numpy()) for c, o in zip(codes, out)) and np.array_equal(z, zo.cpu().numpy())


# codes and latent of 0.1, 1.6, 2.8 MB: by a kernel, and side by side into the ring from 1 MiB on (one by one they were a wait each); 4.2 MB: one by one
@pytest.mark.parametrize("rows,samples,waits", [(1, 30011, 1), (1, 800000, 1), (3, 470001, 1), (4, 522000, 4)])
def test_results_of_an_encode_share_a_wait(snac, rows, samples, waits):
    a = (0.1 * np.random.default_rng(samples).standard_normal((rows, samples))).astype(np.float32)
    codes, z = snac.encode(a, return_latent=True)
    total = z.nbytes + sum(c.nbytes for c in codes)
    assert (total < 4 << 20) == (waits == 1)
    before = _lib.lib().mis_debug_result_waits()
    again, z2 = snac.encode(a, return_latent=True)
    assert _lib.lib().mis_debug_result_waits() - before == waits
    assert np.array_equal(z, z2) and all(np.array_equal(x, y) for x, y in zip(codes, again))


@pytest.mark.parametrize("rows,frames", [(1, 1), (1, 30), (1, 251), (3, 250), (4, 400), (1, 1400)])
def test_dac_decode(dac, rows, frames):
    rng = np.random.default_rng(frames)
    codes = rng.integers(0, 1024, (rows, dac.config.n_codebooks, frames)).astype(np.int32)
    host = dac.decode_from_codes(codes)
    on = torch.from_numpy(codes).cuda()
    out = torch.zeros(host.shape, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    assert _lib.lib().mis_dac_decode_codes(dac._h, on.data_ptr(), rows, frames, out.data_ptr()) == 0
    assert np.array_equal(host, out.cpu().numpy()) and np.abs(host).max() > 0
