"""What Whisper's entry points take: rows much longer than a window, device memory that work on the default stream still writes or reads, more rows than memory."""
import ctypes as C

import numpy as np
import pytest
import torch

import mlx_audio_swift_amd as mas
from mlx_audio_swift_amd import _lib
from mlx_audio_swift_amd.generation import AudioGenerationError, check
from oracle import whisper as owhisper

pytestmark = pytest.mark.gpu


def model():
    ocfg = owhisper.TINY
    return ocfg, mas.WhisperModel.from_weights(mas.WhisperConfig(**{k: getattr(ocfg, k) for k in ocfg.__dataclass_fields__}), owhisper.make_synthetic_weights(ocfg, seed=5))


def generate(dev, pcm_ptr, lens, stride, n=6):
    """mis_stt_whisper_generate on a pointer: rows of `stride` samples, `lens` of them valid."""
    B = len(lens)
    lens = np.asarray(lens, np.int64)
    prompt = np.asarray([3, 5], np.int32)
    sp = _lib.SttParamsC(n, 0.0, 0, dev.config.vocab_size - 1, dev.config.vocab_size - 1, None, 0, None, 0)
    toks, ts, nt = C.c_void_p(), C.c_int64(), (C.c_int32 * B)()
    check(_lib.lib().mis_stt_whisper_generate(dev._h, pcm_ptr, lens.ctypes.data, B, stride, prompt.ctypes.data, 2, C.byref(sp), C.byref(toks), C.byref(ts), nt))
    arr = np.ctypeslib.as_array(C.cast(toks, C.POINTER(C.c_int32)), shape=(B, max(ts.value, 1)))
    out = [arr[b, :nt[b]].tolist() for b in range(B)]
    _lib.lib().mis_free(toks)
    return out


def test_samples_past_the_window_are_not_copied():
    """Rows of 160 MB of which 3 s, and more than a window, are valid: no device memory for the rest, and the ids of rows cut to the window."""
    ocfg, dev = model()
    rng = np.random.default_rng(2)
    lens, stride = [48000, 600000], 40_000_000
    pcm = np.zeros((2, stride), np.float32)
    for b, n in enumerate(lens):
        pcm[b, :n] = 0.1 * rng.standard_normal(n)
    short = np.ascontiguousarray(pcm[:, :480000])
    ref = generate(dev, short.ctypes.data, [48000, 480000], 480000)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    assert generate(dev, pcm.ctypes.data, lens, stride) == ref
    assert free - torch.cuda.mem_get_info()[0] < 32 << 20


def busy():
    """Queue tens of milliseconds of work on the default stream."""
    a = torch.ones(8192, 8192, device="cuda", dtype=torch.bfloat16)
    b = torch.zeros_like(a)
    for _ in range(60):
        torch.mm(a, a, out=b)


def test_device_memory_is_read_and_written_in_the_order_of_the_default_stream():
    ocfg, dev = model()
    rng = np.random.default_rng(3)
    feats = rng.standard_normal((9, 3000, ocfg.num_mel_bins)).astype(np.float32)          # 8.6 MB: past the size where host memory takes the ring
    pcm = (0.1 * rng.standard_normal((9, 480000))).astype(np.float32)
    want, ids = dev.encode(feats), generate(dev, pcm.ctypes.data, [480000] * 9, 480000)
    src_f, src_p = torch.from_numpy(feats).cuda(), torch.from_numpy(pcm).cuda()
    f, p = torch.zeros_like(src_f), torch.zeros_like(src_p)
    out = torch.full((9, 1500, ocfg.d_model), 7.0, device="cuda")
    torch.cuda.synchronize()
    busy()
    f.copy_(src_f)                                                 # queued behind it, as is the reader of the old output
    old = out.clone()
    check(_lib.lib().mis_whisper_encode(dev._h, f.data_ptr(), 9, out.data_ptr()))
    assert np.array_equal(out.cpu().numpy(), want) and bool((old == 7.0).all())
    busy()
    p.copy_(src_p)
    assert generate(dev, p.data_ptr(), [480000] * 9, 480000) == ids


def test_an_allocation_that_fails_leaves_no_half_made_state():
    """64 rows of 2 million decoder positions in 16 layers would be 1 TB of caches: refused each time, and one row still runs."""
    ocfg = owhisper.TINY
    cfg = mas.WhisperConfig(**{**{k: getattr(ocfg, k) for k in ocfg.__dataclass_fields__}, "decoder_layers": 16, "max_target_positions": 2_000_000})
    dev = mas.WhisperModel.synthetic(cfg)
    feats = np.random.default_rng(4).standard_normal((64, 3000, ocfg.num_mel_bins)).astype(np.float32)
    for _ in range(2):
        with pytest.raises(AudioGenerationError):
            dev.encode(feats, want_output=False)
    with pytest.raises(AudioGenerationError):
        dev.decoder_forward(np.zeros(64, np.int32))
    assert np.isfinite(dev.encode(feats[:1])).all()
