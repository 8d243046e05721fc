"""Workloads of the engine as a user's program runs them: text-to-speech generation with the SNAC codec behind it, prompt passes, codec
encode / decode, speech recognition.  Everything goes through the Python mirror of the C ABI (host arrays in, host arrays out, as the
mirror takes and returns them); weights are synthetic, seeded, and of the configurations that the tests and bench.py use.

So that tokens can be compared between two correct implementations, the synthetic language models predict with the confidence of a trained
one: the output projection's row of token pi(t) points along the embedding of t (speech model), the decoder's position embedding p points along
the embedding of the token that follows (Whisper).  Every layer runs on ordinary random weights."""
import math

import numpy as np
import torch

import mlx_audio_swift_amd as mas

DEV = "cuda"
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64

# ------------------------------------------------------------------------------------------------------------------------ the cases

SIZES = {  # Whisper: the smallest and the largest configuration of the family that the tests run
    "tiny": dict(vocab_size=51865, num_mel_bins=80, d_model=384, encoder_layers=4, encoder_attention_heads=6, encoder_ffn_dim=1536,
                 decoder_layers=4, decoder_attention_heads=6, decoder_ffn_dim=1536),
    "large": dict(vocab_size=51866, num_mel_bins=128, d_model=1280, encoder_layers=32, encoder_attention_heads=20, encoder_ffn_dim=5120,
                  decoder_layers=32, decoder_attention_heads=20, decoder_ffn_dim=5120),
}


def listed():
    return [
        # one short utterance of codes to samples: what a streaming player asks for, 1 s of audio
        dict(name="snac_decode_1x12", kind="snac_decode", rows=1, groups=12),
        # a whole batch of long utterances: the codec behind a batch-32 generation, 8.2 s a row
        dict(name="snac_decode_32x96", kind="snac_decode", rows=32, groups=96),
        # a reference recording to codes: the first half of voice cloning, 6.3 s, not a multiple of the frame
        dict(name="snac_encode_1x151k", kind="snac_encode", rows=1, samples=151111),
        # the 16 kHz Descript codec, 250 frames = 5 s
        dict(name="dac_decode_1x250", kind="dac_decode", rows=1, frames=250),
        # speech recognition of one window with the smallest model: all latency
        dict(name="whisper_tiny_1", kind="transcribe", size="tiny", rows=1, seconds=11.0, tokens=40),
        # a recording of four minutes in eight windows with the largest model
        dict(name="whisper_large_8", kind="transcribe", size="large", rows=8, seconds=30.0, tokens=40),
        # the encoder alone (features for alignment or language identification)
        dict(name="whisper_encode_8", kind="whisper_encode", size="large", rows=8),
        # one listener: a short sentence at batch 1
        dict(name="tts_1", kind="tts", rows=1, prompt=24, frames=10, bits=0),
        # the served batch: 32 sentences
        dict(name="tts_32", kind="tts", rows=32, prompt=32, frames=12, bits=0),
        # the 8-bit checkpoint, as most users download it, with a few sentences at once
        dict(name="tts_5_q8", kind="tts", rows=5, prompt=41, frames=10, bits=8),
        # voice-cloning prompts (reference codes and transcript) of eight callers before their first token
        dict(name="prefill_8x450", kind="prefill", rows=8, prompt=450),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["snac_decode", "snac_decode", "snac_encode", "dac_decode", "transcribe", "whisper_encode", "tts", "tts", "prefill"])
    if kind == "snac_decode":
        return dict(kind=kind, rows=_log(rng, 1, 32), groups=_log(rng, 4, 96))
    if kind == "snac_encode":
        return dict(kind=kind, rows=_log(rng, 1, 4), samples=_log(rng, 12000, 240000))
    if kind == "dac_decode":
        return dict(kind=kind, rows=_log(rng, 1, 4), frames=_log(rng, 30, 400))
    if kind == "transcribe":
        return dict(kind=kind, size=rng.choice(["tiny", "large"]), rows=_log(rng, 1, 8), seconds=round(rng.uniform(2.0, 30.0), 2), tokens=_log(rng, 10, 40))
    if kind == "whisper_encode":
        return dict(kind=kind, size=rng.choice(["tiny", "large"]), rows=_log(rng, 1, 8))
    if kind == "tts":
        return dict(kind=kind, rows=_log(rng, 1, 32), prompt=_log(rng, 12, 120), frames=_log(rng, 3, 10), bits=rng.choice([0, 0, 8]))
    rows = _log(rng, 1, 16)
    return dict(kind=kind, rows=rows, prompt=_log(rng, 30, min(900, 3600 // rows)))


# ------------------------------------------------------------------------------------------------------------- inputs made from a seed

class Make:
    """Values in a fixed order from one seed, on the GPU."""

    def __init__(self, seed, part):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1000003 * int(seed) + part)

    def uniform(self, shape, amp, dtype=F32, mid=0.0):
        return torch.empty(tuple(shape), dtype=dtype, device=DEV).uniform_(-amp, amp, generator=self.g).add_(mid)

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, tuple(shape), generator=self.g, device=DEV)

    def speech(self, rows, n, rate):
        """Harmonics of a gliding pitch under a syllable envelope, and a little noise."""
        t = torch.arange(n, device=DEV, dtype=F64) / rate
        pitch, glide = self.uniform((rows, 1), 60.0, F64, 160.0), self.uniform((rows, 1), 25.0, F64)
        phase = 2 * math.pi * (pitch * t + glide * torch.sin(2 * math.pi * 0.7 * t))
        x = sum(torch.sin(k * phase + float(k)) / k for k in range(1, 9))
        env = 0.55 + 0.45 * torch.sin(2 * math.pi * self.uniform((rows, 1), 1.0, F64, 4.0) * t)
        return (0.12 * x * env + self.uniform((rows, n), 0.01, F64)).to(F32)


def snac_config():
    return mas.SNACConfig()


def snac_weights(seed, encoder):
    """SNAC 24 kHz in the checkpoint's layout, weight-norm pairs included; activations stay of order one."""
    cf, m, W = snac_config(), Make(seed, 1), {}
    latent = cf.encoder_dim * 2 ** len(cf.encoder_rates)

    def wn(p, out, k, per, gain=1.0, bias=True):
        v = m.uniform((out, k, per), gain * math.sqrt(3.0 / (per * k)))
        W[p + ".weight_v"] = v
        W[p + ".weight_g"] = v.pow(2).sum((1, 2), keepdim=True).sqrt() * m.uniform((out, 1, 1), 0.3, mid=1.0)
        if bias:
            W[p + ".bias"] = m.uniform((out,), 0.1)

    def unit(r, c):
        W[r + ".0.alpha"] = m.uniform((1, c, 1), 0.7, mid=1.25)
        wn(r + ".1", c, 7, 1)
        W[r + ".2.alpha"] = m.uniform((1, c, 1), 0.7, mid=1.25)
        wn(r + ".3", c, 1, c, 0.2)

    for i in range(len(cf.vq_strides)):
        p = "quantizer.quantizers.%d" % i
        W[p + ".codebook.weight"] = m.uniform((cf.codebook_size, cf.codebook_dim), math.sqrt(3.0))
        wn(p + ".in_proj", cf.codebook_dim, 1, latent)
        wn(p + ".out_proj", latent, 1, cf.codebook_dim)
    p = "decoder.model.layers"
    wn(p + ".0", latent, 7, 1)
    wn(p + ".1", cf.decoder_dim, 1, latent)
    for i, s in enumerate(cf.decoder_rates):
        a, b = cf.decoder_dim >> i, cf.decoder_dim >> (i + 1)
        q = "%s.%d.block.layers" % (p, 2 + i)
        W[q + ".0.alpha"] = m.uniform((1, a, 1), 0.7, mid=1.25)
        wn(q + ".1", a, 2 * s, b)
        W[q + ".1.weight_v"] *= math.sqrt(s * b / a)                                                       # two taps of each input reach one output
        W[q + ".1.weight_g"] *= math.sqrt(s * b / a)
        W[q + ".1.bias"] = m.uniform((b,), 0.1)
        wn(q + ".2.linear", b, 1, b, 0.3, bias=False)
        for j in range(3):
            unit("%s.%d.block.layers" % (q, 3 + j), b)
    n, last = 2 + len(cf.decoder_rates), cf.decoder_dim >> len(cf.decoder_rates)
    W["%s.%d.alpha" % (p, n)] = m.uniform((1, last, 1), 0.7, mid=1.25)
    wn("%s.%d" % (p, n + 1), 1, 7, last, 0.12)
    if encoder:
        e, c = "encoder.block.layers", cf.encoder_dim
        wn(e + ".0", c, 7, 1, 3.0)
        for i, s in enumerate(cf.encoder_rates):
            q = "%s.%d.block.layers" % (e, 1 + i)
            for j in range(3):
                unit("%s.%d.block.layers" % (q, j), c)
            W[q + ".3.alpha"] = m.uniform((1, c, 1), 0.7, mid=1.25)
            wn(q + ".4", 2 * c, 2 * s, c)
            c *= 2
        wn("%s.%d" % (e, 1 + len(cf.encoder_rates)), c, 7, 1)
    return W


def snac_codes(seed, rows, groups):
    m = Make(seed, 2)
    return [m.ints(0, 4096, (rows, groups * k)) for k in (1, 2, 4)]


def dac_config():
    return mas.DescriptDACConfig()


def dac_weights(seed):
    cf, m, W = dac_config(), Make(seed, 3), {}

    def wn(p, out, k, per, gain=1.0, transposed=False):
        v = m.uniform((out, k, per), gain * math.sqrt(3.0 / (k * per)))
        dims, shape = ((0, 1), (1, 1, per)) if transposed else ((1, 2), (out, 1, 1))
        W[p + ".weight_v"] = v
        W[p + ".weight_g"] = v.pow(2).sum(dims, keepdim=True).sqrt() * m.uniform(shape, 0.3, mid=1.0)
        W[p + ".bias"] = m.uniform((out,), 0.05)

    for i in range(cf.n_codebooks):
        p = "quantizer.quantizers.%d" % i
        W[p + ".codebook.weight"] = m.uniform((cf.codebook_size, cf.codebook_dim), math.sqrt(3.0 / cf.n_codebooks))
        wn(p + ".outProj", cf.resolved_latent, 1, cf.codebook_dim)
    wn("decoder.model.0", cf.decoder_dim, 7, cf.resolved_latent)
    for i, s in enumerate(cf.decoder_rates):
        a, b = cf.decoder_dim >> i, cf.decoder_dim >> (i + 1)
        p = "decoder.model.%d.block" % (i + 1)
        W[p + ".0.alpha"] = m.uniform((1, 1, a), 0.7, mid=1.25)
        wn(p + ".1", b, 2 * s, a, 0.8 * math.sqrt(s), transposed=True)
        for j in range(3):
            q = "%s.%d.block" % (p, j + 2)
            W[q + ".0.alpha"] = m.uniform((1, 1, b), 0.7, mid=1.25)
            wn(q + ".1", b, 7, b, 0.7)
            W[q + ".2.alpha"] = m.uniform((1, 1, b), 0.7, mid=1.25)
            wn(q + ".3", b, 1, b, 0.3)
    n, last = len(cf.decoder_rates), cf.decoder_dim >> len(cf.decoder_rates)
    W["decoder.model.%d.alpha" % (n + 1)] = m.uniform((1, 1, last), 0.7, mid=1.25)
    wn("decoder.model.%d" % (n + 2), 1, 7, last, 0.5)
    return W


# ---- the 3B speech model (the configuration of bench.py, with an output projection of its own)

SPEECH0, SLOT, END_OF_SPEECH = 128266, 4096, 128258   # first audio token; a frame is seven slots of 4096 codes
LM = dict(hidden_size=3072, num_hidden_layers=28, intermediate_size=8192, num_attention_heads=24, num_key_value_heads=8, head_dim=128, vocab_size=156940,
          rms_norm_eps=1e-5, rope_theta=500000.0, tie_word_embeddings=False)
ROPE = dict(factor=32.0, low_freq_factor=1.0, high_freq_factor=4.0, original_max_position_embeddings=8192, rope_type="llama3")


def following(seed):
    """pi on the audio tokens: slot k to slot k + 1, codes permuted."""
    r = np.random.default_rng(int(seed) + 17)
    a, b, c = 2 * r.integers(1, 2048, 7) + 1, r.integers(0, SLOT, 7), np.arange(SLOT)
    return np.concatenate([SPEECH0 + ((k + 1) % 7) * SLOT + (a[k] * c + b[k]) % SLOT for k in range(7)])


def lm_weights(seed, bits):
    """(name, tensor) or (name, (codes, scales, biases)) one after the other: a caller need not hold them all."""
    d, ff, L, V = LM["hidden_size"], LM["intermediate_size"], LM["num_hidden_layers"], LM["vocab_size"]
    q, kv, m = LM["num_attention_heads"] * LM["head_dim"], LM["num_key_value_heads"] * LM["head_dim"], Make(seed, 4)
    emb = m.uniform((V, d), math.sqrt(3.0), BF)
    yield "model.embed_tokens.weight", emb
    head = m.uniform((V, d), 2 * math.sqrt(3.0 / d), BF)
    head[torch.from_numpy(following(seed)).to(DEV)] = emb[SPEECH0:SPEECH0 + 7 * SLOT] * (2 / math.sqrt(d))
    yield "lm_head.weight", head
    del emb, head
    yield "model.norm.weight", m.uniform((d,), 0.1, BF, 1.0)
    for li in range(L):
        p = "model.layers.%d" % li
        for n in ("input_layernorm", "post_attention_layernorm"):
            yield "%s.%s.weight" % (p, n), m.uniform((d,), 0.1, BF, 1.0)
        for n, out, per, gain in (("self_attn.q_proj", q, d, 1.2), ("self_attn.k_proj", kv, d, 1.2), ("self_attn.v_proj", kv, d, 1.0),
                                  ("self_attn.o_proj", d, q, 0.3), ("mlp.gate_proj", ff, d, 1.0), ("mlp.up_proj", ff, d, 1.0), ("mlp.down_proj", d, ff, 0.25)):
            amp = gain * math.sqrt(3.0 / per)
            if bits:
                codes = m.ints(0, 256, (out, per)).to(torch.uint8)
                grain = m.uniform((out, per // 64), 0.2, F32, 1.0) * amp
                yield "%s.%s.weight" % (p, n), (codes, (grain * (2.0 / 255.0)).to(BF), (-grain).to(BF))
            else:
                yield "%s.%s.weight" % (p, n), m.uniform((out, per), amp, BF)


def prompts(seed, rows, n):
    """Ragged rows: a text, the start of speech, and the frame that the speech goes on from."""
    r = np.random.default_rng(int(seed) + 29)
    out = []
    for b in range(rows):
        k = max(1, n - 11 - (int(r.integers(0, max(1, n // 4))) if b else 0))
        frame = SPEECH0 + np.arange(7) * SLOT + r.integers(0, SLOT, 7)
        out.append(np.concatenate([[128259], r.integers(0, 128000, k), [128009, 128260, 128257], frame]).astype(np.int32))
    return out


def cloning_prompts(seed, rows, n):
    """Ragged rows: the transcript and the codes of a reference recording, then the text."""
    r = np.random.default_rng(int(seed) + 31)
    out = []
    for b in range(rows):
        k = n - (int(r.integers(0, max(1, n // 3))) if b else 0)
        frames = max(1, (k * 2 // 3) // 7)
        codes = (SPEECH0 + np.tile(np.arange(7), frames) * SLOT + r.integers(0, SLOT, 7 * frames))
        text = r.integers(0, 128000, max(2, k - len(codes) - 10))
        h = len(text) // 2
        out.append(np.concatenate([[128259], text[:h], [128009, 128260, 128261, 128257], codes, [128258, 128262, 128259], text[h:], [128009, 128260]]).astype(np.int32))
    return out


# ---- Whisper

START = 50258


def spoken(seed, n):
    """The tokens that the model says, by position of the one before."""
    return np.random.default_rng(int(seed) + 41).integers(300, 50000, n)


def whisper_weights(size, seed, decoder=True):
    cf, m = SIZES[size], Make(seed, 5)
    d, V = cf["d_model"], cf["vocab_size"]

    def lin(p, out, per, gain=1.0, bias=True):
        yield p + ".weight", m.uniform((out, per), gain * math.sqrt(3.0 / per), BF)
        if bias:
            yield p + ".bias", m.uniform((out,), 0.05, BF)

    def norm(p):
        yield p + ".weight", m.uniform((d,), 0.1, BF, 1.0)
        yield p + ".bias", m.uniform((d,), 0.05, BF)

    def attn(p):
        yield from lin(p + ".q_proj", d, d, 1.2)
        yield from lin(p + ".k_proj", d, d, 1.2, False)
        yield from lin(p + ".v_proj", d, d)
        yield from lin(p + ".out_proj", d, d, 0.3)

    e = "model.encoder"
    yield e + ".conv1.weight", m.uniform((d, cf["num_mel_bins"], 3), math.sqrt(1.0 / cf["num_mel_bins"]), BF)
    yield e + ".conv1.bias", m.uniform((d,), 0.05, BF)
    yield e + ".conv2.weight", m.uniform((d, d, 3), math.sqrt(3.0 / d), BF)
    yield e + ".conv2.bias", m.uniform((d,), 0.05, BF)
    yield e + ".embed_positions.weight", m.uniform((1500, d), 0.5, BF)
    for li in range(cf["encoder_layers"]):
        p = "%s.layers.%d" % (e, li)
        yield from attn(p + ".self_attn")
        yield from norm(p + ".self_attn_layer_norm")
        yield from lin(p + ".fc1", cf["encoder_ffn_dim"], d)
        yield from lin(p + ".fc2", d, cf["encoder_ffn_dim"], 0.3)
        yield from norm(p + ".final_layer_norm")
    yield from norm(e + ".layer_norm")
    e = "model.decoder"
    emb = m.uniform((V, d), 0.5, BF)
    yield e + ".embed_tokens.weight", emb
    yield e + ".embed_positions.weight", (emb[torch.from_numpy(spoken(seed, 448)).to(DEV)].to(F32) * 3.0).to(BF)
    for li in range(cf["decoder_layers"]):
        p = "%s.layers.%d" % (e, li)
        yield from attn(p + ".self_attn")
        yield from norm(p + ".self_attn_layer_norm")
        yield from attn(p + ".encoder_attn")
        yield from norm(p + ".encoder_attn_layer_norm")
        yield from lin(p + ".fc1", cf["decoder_ffn_dim"], d)
        yield from lin(p + ".fc2", d, cf["decoder_ffn_dim"], 0.3)
        yield from norm(p + ".final_layer_norm")
    yield from norm(e + ".layer_norm")


def windows(case, seed):
    """Recordings of up to 30 s; all but the first a little shorter."""
    n = int(16000 * case["seconds"])
    x = Make(seed, 6).speech(case["rows"], n, 16000.0)
    r = np.random.default_rng(int(seed) + 43)
    return [x[b, : n - (int(r.integers(0, 4000)) if b else 0)] for b in range(case["rows"])]


def log_mel(x, n_mels):
    """Whisper's features of one window in 64 bits: [3000, n_mels]."""
    x = torch.nn.functional.pad(x.to(F64), (0, 480000 - x.shape[0]))
    x = torch.cat([x[1:201].flip(0), x, x[-201:-1].flip(0)])
    w = 0.5 - 0.5 * torch.cos(2 * math.pi * torch.arange(400, device=x.device, dtype=F64) / 400)
    power = torch.fft.rfft(x.unfold(0, 400, 160) * w).abs().pow(2)[:-1]
    hz = np.arange(201) * 40.0
    m = np.linspace(0.0, 15.0 + 27.0 * math.log(8.0) / math.log(6.4), n_mels + 2)
    f = np.where(m < 15.0, m * 200.0 / 3.0, 1000.0 * np.exp(np.log(6.4) / 27.0 * (m - 15.0)))
    up, down = (hz[:, None] - f[None, :-2]) / (f[1:-1] - f[:-2]), (f[None, 2:] - hz[:, None]) / (f[2:] - f[1:-1])
    bank = np.maximum(0.0, np.minimum(up, down)) * (2.0 / (f[2:] - f[:-2]))
    s = (power @ torch.from_numpy(bank).to(x.device)).clamp_min(1e-10).log10()
    return (torch.maximum(s, s.max() - 8.0) + 4.0) / 4.0


def encoder_features(case, seed):
    n_mels = SIZES[case["size"]]["num_mel_bins"]
    x = Make(seed, 7).speech(case["rows"], 480000, 16000.0)
    return torch.stack([log_mel(r, n_mels) for r in x]).to(F32)


# ------------------------------------------------------------------------------------------------------------------------- prepare, run

def host(x):
    return x.cpu().numpy()


def make_snac(seed, encoder=False):
    return mas.SNAC.from_weights(snac_config(), {k: v.cpu() for k, v in snac_weights(seed, encoder).items()})


def make_lm(seed, bits, codec):
    lm = mas.LlamaTTSModel(mas.LlamaTTSConfiguration(rope_scaling=dict(ROPE), **LM), codec)
    for name, t in lm_weights(seed, bits):
        if isinstance(t, tuple):
            torch.cuda.synchronize()
            codes, sc, bi = t
            mas.generation.check(mas._lib.lib().mis_tts_set_tensor_quantized(lm._h, name.encode(), codes.data_ptr(), sc.data_ptr(), bi.data_ptr(), mas._lib.MIS_BF16,
                                                                             codes.shape[0], codes.shape[1], 64, 8))
        else:
            torch.cuda.synchronize()
            lm.set_tensor(name, t)
    lm.finalize()
    return lm


def make_whisper(size, seed):
    m = mas.WhisperModel(mas.WhisperConfig(**SIZES[size]))
    for name, t in whisper_weights(size, seed):
        torch.cuda.synchronize()
        m.set_tensor(name, t)
    m.finalize()
    return m


def prepare(case, seed):
    k, st = case["kind"], dict(case=case)
    if k == "snac_decode":
        st["codec"] = make_snac(seed)
        st["codec"].set_noise(False, seed)
        st["codes"] = [host(c).astype(np.int32) for c in snac_codes(seed, case["rows"], case["groups"])]
    elif k == "snac_encode":
        st["codec"] = make_snac(seed, True)
        st["audio"] = host(Make(seed, 8).speech(case["rows"], case["samples"], 24000.0))
    elif k == "dac_decode":
        cf = dac_config()
        st["codec"] = mas.DescriptDAC.from_weights(cf, {n: v.cpu() for n, v in dac_weights(seed).items()})
        st["codes"] = host(Make(seed, 9).ints(0, cf.codebook_size, (case["rows"], cf.n_codebooks, case["frames"]))).astype(np.int32)
    elif k == "transcribe":
        st["model"] = make_whisper(case["size"], seed)
        st["windows"] = [host(w) for w in windows(case, seed)]
        st["params"] = mas.STTGenerateParameters(max_tokens=case["tokens"], temperature=0.0, eot_id=50257, timestamp_begin=50364)
    elif k == "whisper_encode":
        st["model"] = make_whisper(case["size"], seed)
        st["features"] = host(encoder_features(case, seed))
    elif k == "tts":
        st["codec"] = make_snac(seed)
        st["model"] = make_lm(seed, case["bits"], st["codec"])
        st["prompts"] = prompts(seed, case["rows"], case["prompt"])
        st["params"] = mas.GenerateParameters(max_tokens=7 * case["frames"], seed=seed)
    elif k == "prefill":
        st["model"] = make_lm(seed, 0, None)
        st["prompts"] = cloning_prompts(seed, case["rows"], case["prompt"])
    return st


PROMPT = [START, 50259, 50359, 50363]


def run(st):
    k = st["case"]["kind"]
    if k == "snac_decode":
        return st["codec"].decode(st["codes"])
    if k == "snac_encode":
        codes, z = st["codec"].encode(st["audio"], return_latent=True)
        return dict(codes=codes, z=z)
    if k == "dac_decode":
        return st["codec"].decode_from_codes(st["codes"])
    if k == "transcribe":
        m, n = st["model"], st["case"]["rows"]
        ids = m.transcribe_windows(st["windows"], PROMPT, st["params"])
        m.decoder_reset()                                                     # the windows are still encoded: the model's view of the first token
        return dict(tokens=np.asarray(ids, np.int32), logits=m.decoder_forward([START] * n))
    if k == "whisper_encode":
        return st["model"].encode(st["features"])
    if k == "tts":
        pcm, tokens = st["model"].generate_batch(st["prompts"], st["params"], return_tokens=True)
        logits = st["model"].lm_forward([END_OF_SPEECH] * len(tokens))         # the rows stand behind their tokens: what follows the end of speech
        return dict(pcm=np.stack(pcm), tokens=np.stack(tokens), logits=logits)
    return st["model"].lm_prefill(st["prompts"])


# --------------------------------------------------------------------------------------------------------------------------------- work

def _snac_decoder_macs(T0):
    cf = snac_config()
    latent = cf.encoder_dim * 2 ** len(cf.encoder_rates)
    macs, weights, T, c = T0 * (7 * latent + latent * cf.decoder_dim), 3 * cf.codebook_size * cf.codebook_dim + latent * (7 + cf.decoder_dim), T0, cf.decoder_dim
    for s in cf.decoder_rates:
        T, b = T * s, c // 2
        macs += T * (2 * c * b + b * b + 3 * (7 * b + b * b))
        weights += c * 2 * s * b + b * b + 3 * (7 * b + b * b)
        c = b
    return macs + T * 7 * c, weights, T


def _lm_counts(bits):
    d, ff, q, kv = LM["hidden_size"], LM["intermediate_size"], LM["num_attention_heads"] * LM["head_dim"], LM["num_key_value_heads"] * LM["head_dim"]
    per = LM["num_hidden_layers"] * (d * (2 * q + 2 * kv) + 3 * d * ff)
    return per, per * (1.0625 if bits else 2.0), 2.0 * LM["vocab_size"] * d, LM["num_hidden_layers"] * 2 * kv * 2.0


def work(case):
    k, rows = case["kind"], case["rows"]
    if k == "snac_decode":
        macs, w, n = _snac_decoder_macs(4 * case["groups"])
        return dict(bytes=4.0 * (w + rows * (n + 7 * case["groups"])), flops=2.0 * rows * macs)
    if k == "snac_encode":
        cf = snac_config()
        T = -(-case["samples"] // 2048) * 2048
        macs, w, c, t = 7 * cf.encoder_dim * T, 0, cf.encoder_dim, T
        for s in cf.encoder_rates:
            macs += t * 3 * (7 * c + c * c) + t // s * (2 * c * 2 * s * c)
            w += 3 * (7 * c + c * c) + 2 * c * 2 * s * c
            t, c = t // s, 2 * c
        macs += t * c * (7 + 3 * 8 * 2) + t * 2 * 4096 * 8
        return dict(bytes=4.0 * (w + rows * (case["samples"] + t * c + t * 2)), flops=2.0 * rows * macs)
    if k == "dac_decode":
        cf = dac_config()
        T, c = case["frames"], cf.decoder_dim
        w = cf.resolved_latent * 7 * c
        macs = T * w
        for s in cf.decoder_rates:
            T, b = T * s, c // 2
            macs += T * (2 * c * b + 3 * 8 * b * b)
            w += 2 * s * c * b + 3 * 8 * b * b
            c = b
        return dict(bytes=4.0 * (w + rows * (T + case["frames"] * cf.n_codebooks)), flops=2.0 * rows * (macs + T * 7 * c))
    if k in ("transcribe", "whisper_encode"):
        cf = SIZES[case["size"]]
        d, f, L, V = cf["d_model"], cf["encoder_ffn_dim"], cf["encoder_layers"], cf["vocab_size"]
        enc = L * (4 * d * d + 2 * d * f)
        flops = rows * (2.0 * 1500 * enc + 4.0 * L * 1500 * 1500 * d + 2 * 3 * cf["num_mel_bins"] * d * 3000 + 2 * 3 * d * d * 1500)
        if k == "whisper_encode":
            return dict(bytes=2.0 * enc + 4.0 * rows * (3000 * cf["num_mel_bins"] + 1500 * d), flops=flops)
        dec, steps = L * (6 * d * d + 2 * d * f), len(PROMPT) + case["tokens"]
        flops += rows * (2.0 * steps * dec + 2.0 * case["tokens"] * V * d + 4.0 * L * 1500 * d * d + steps * L * 4.0 * 1500 * d)
        return dict(bytes=2.0 * enc + 4.0 * rows * 16000 * case["seconds"] + steps * (2.0 * dec + rows * L * 1500 * d * 4.0) + case["tokens"] * 2.0 * V * d, flops=flops)
    if k == "tts":
        per, wb, hb, kvb = _lm_counts(case["bits"])
        steps, n = 7 * case["frames"], case["prompt"]
        macs, w, N = _snac_decoder_macs(4 * (case["frames"] + 1))
        return dict(bytes=(steps + 1) * (wb + hb) + rows * kvb * steps * (n + steps / 2.0) + 4.0 * (w + rows * N) + 4.0 * rows * LM["vocab_size"],
                    flops=2.0 * rows * ((n + steps) * per + steps * LM["vocab_size"] * LM["hidden_size"] + macs))
    per, wb, hb, kvb = _lm_counts(0)
    n = 0.85 * case["prompt"]
    return dict(bytes=wb + hb + rows * (kvb * n + 4.0 * LM["vocab_size"]), flops=2.0 * rows * (n * per + LM["vocab_size"] * LM["hidden_size"]))


def tolerance(case):
    if case["kind"] in ("snac_decode", "dac_decode"):
        return {"rel": 1e-4, "max": 0.01}                     # split-bf16 products: 2.2e-5 from 64 bits
    if case["kind"] == "snac_encode":
        return {"rel": 1e-4, "max": 0.01, "differ": 0.01}
    return {"rel": 0.03, "max": 0.5, "differ": 0.0}      # bf16 through up to 32 layers: 0.012 to 0.016 from 64 bits on each side


# ------------------------------------------------------------------------------------------------------- the same in 64 bits, plain torch

def conv(x, w, b=None, stride=1, pad=0, dil=1):
    """x [B, I, T], w [O, K, I] ([O, K, 1] for one channel each)."""
    x = torch.nn.functional.pad(x, (pad, pad))
    K = w.shape[1]
    n = (x.shape[2] - dil * (K - 1) - 1) // stride + 1
    y = 0
    for k in range(K):
        s = x[:, :, k * dil: k * dil + (n - 1) * stride + 1: stride]
        y = y + (w[:, k, 0][None, :, None] * s if w.shape[2] == 1 and x.shape[1] == w.shape[0] and x.shape[1] > 1 else torch.matmul(w[:, k].contiguous(), s.contiguous()))
    return y if b is None else y + b[None, :, None]


def conv_transposed(x, w, b, stride, pad, extra):
    """x [B, I, T], w [I, K, O]: `pad` samples dropped on the left, pad - extra on the right."""
    B, _, T = x.shape
    K, O = w.shape[1], w.shape[2]
    y = torch.zeros(B, O, (T - 1) * stride + K, dtype=x.dtype, device=x.device)
    for k in range(K):
        y[:, :, k: k + (T - 1) * stride + 1: stride] += torch.matmul(w[:, k].t().contiguous(), x)
    return y[:, :, pad: y.shape[2] - pad + extra] + b[None, :, None]


def snake(x, a):
    a = a.reshape(1, -1, 1)
    return x + torch.sin(a * x).pow(2) / (a + 1e-9)


class Codec64:
    def __init__(self, weights):
        self.w = {k: v.to(F64) for k, v in weights.items()}

    def wn(self, p, dims=(1, 2)):
        g, v = self.w[p + ".weight_g"], self.w[p + ".weight_v"]
        return g * v / (v.pow(2).sum(dims, keepdim=True).sqrt() + 1e-12)

    def conv(self, p, x, **kw):
        return conv(x, self.wn(p), self.w.get(p + ".bias"), **kw)

    def unit(self, p, x, dil, sep=""):
        h = self.conv(p + ".1", snake(x, self.w[p + ".0.alpha"]), pad=3 * dil, dil=dil)
        return x + self.conv(p + ".3", snake(h, self.w[p + ".2.alpha"]))


def _mix64(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def codec_noise(seed, block, rows, n):
    """The codec's documented counter generator: Box-Muller on 24-bit uniforms keyed by (seed, block, row, sample)."""
    with np.errstate(over="ignore"):
        key = _mix64(np.array([int(seed) + 0x51AC0000 + block], np.uint64))
        u = _mix64((key ^ (np.arange(rows, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)))[:, None] + np.arange(n, dtype=np.uint64)[None, :])
    u1 = ((u >> np.uint64(40)).astype(np.float32) + np.float32(0.5)).astype(np.float64) * 2.0 ** -24
    u2 = (((u >> np.uint64(16)) & np.uint64(0xFFFFFF)).astype(np.float32) + np.float32(0.5)).astype(np.float64) * 2.0 ** -24
    return torch.from_numpy(np.sqrt(-2.0 * np.log(u1)) * np.cos(2.0 * np.pi * u2)).to(DEV)


def snac_decode64(weights, codes, seed):
    """codes: three [B, T_i]; [B, 1, N]."""
    cf, c = snac_config(), Codec64(weights)
    z = 0
    for i, s in enumerate(cf.vq_strides):
        p = "quantizer.quantizers.%d" % i
        z = z + c.conv(p + ".out_proj", c.w[p + ".codebook.weight"][codes[i]].transpose(1, 2)).repeat_interleave(s, dim=2)
    p = "decoder.model.layers"
    x = c.conv(p + ".1", c.conv(p + ".0", z, pad=3))
    for i, s in enumerate(cf.decoder_rates):
        q = "%s.%d.block.layers" % (p, 2 + i)
        x = conv_transposed(snake(x, c.w[q + ".0.alpha"]), c.wn(q + ".1"), c.w[q + ".1.bias"], s, -(-s // 2), 0)
        x = x + codec_noise(seed, i, x.shape[0], x.shape[2])[:, None] * c.conv(q + ".2.linear", x)
        for j, dil in enumerate((1, 3, 9)):
            x = c.unit("%s.%d.block.layers" % (q, 3 + j), x, dil)
    n = 2 + len(cf.decoder_rates)
    return torch.tanh(c.conv("%s.%d" % (p, n + 1), snake(x, c.w["%s.%d.alpha" % (p, n)]), pad=3))


def snac_encode64(weights, audio):
    cf, c = snac_config(), Codec64(weights)
    hop = math.prod(cf.encoder_rates) * cf.vq_strides[0]
    x = torch.nn.functional.pad(audio.to(F64), (0, -audio.shape[1] % hop))[:, None]
    p = "encoder.block.layers"
    x = c.conv(p + ".0", x, pad=3)
    for i, s in enumerate(cf.encoder_rates):
        q = "%s.%d.block.layers" % (p, 1 + i)
        for j, dil in enumerate((1, 3, 9)):
            x = c.unit("%s.%d.block.layers" % (q, j), x, dil)
        x = c.conv(q + ".4", snake(x, c.w[q + ".3.alpha"]), stride=s, pad=-(-s // 2))
    z = c.conv("%s.%d" % (p, 1 + len(cf.encoder_rates)), x, pad=3)
    r, codes = z, []
    for i, s in enumerate(cf.vq_strides):
        p = "quantizer.quantizers.%d" % i
        B, C, T = r.shape
        e = c.conv(p + ".in_proj", r.reshape(B, C, T // s, s).mean(3)).transpose(1, 2)
        cb = c.w[p + ".codebook.weight"]
        en, cn = torch.nn.functional.normalize(e, dim=2, eps=1e-12), torch.nn.functional.normalize(cb, dim=1, eps=1e-12)
        idx = (cn.pow(2).sum(1) - 2.0 * torch.matmul(en, cn.t().contiguous())).argmin(2)
        codes.append(idx)
        r = r - c.conv(p + ".out_proj", cb[idx].transpose(1, 2)).repeat_interleave(s, dim=2)
    return codes, z


def dac_decode64(weights, codes):
    cf, c = dac_config(), Codec64(weights)
    x = 0
    for i in range(cf.n_codebooks):
        p = "quantizer.quantizers.%d" % i
        x = x + c.conv(p + ".outProj", c.w[p + ".codebook.weight"][codes[:, i]].transpose(1, 2))
    x = c.conv("decoder.model.0", x, pad=3)
    for i, s in enumerate(cf.decoder_rates):
        p = "decoder.model.%d.block" % (i + 1)
        x = conv_transposed(snake(x, c.w[p + ".0.alpha"]), c.wn(p + ".1", (0, 1)).permute(2, 1, 0), c.w[p + ".1.bias"], s, -(-s // 2), 1)
        for j, dil in enumerate((1, 3, 9)):
            x = c.unit("%s.%d.block" % (p, j + 2), x, dil)
    n = len(cf.decoder_rates)
    return torch.tanh(c.conv("decoder.model.%d" % (n + 2), snake(x, c.w["decoder.model.%d.alpha" % (n + 1)]), pad=3))[:, 0]


def _dequantised(t):
    if not isinstance(t, tuple):
        return t
    codes, sc, bi = (x.to(F64) for x in t)
    return codes * sc.repeat_interleave(64, 1) + bi.repeat_interleave(64, 1)


def lm_logits64(seed, bits, rows):
    """Logits behind the last token of every row (host arrays of ids), [B, V]: one causal pass, each layer's weights made as it is reached."""
    d, H, K, D, eps = LM["hidden_size"], LM["num_attention_heads"], LM["num_key_value_heads"], LM["head_dim"], LM["rms_norm_eps"]
    f = torch.pow(torch.tensor(float(LM["rope_theta"]), dtype=F64), torch.arange(0, D, 2, dtype=F64) / D)
    wl, old = 2 * math.pi * f, ROPE["original_max_position_embeddings"]
    s = (old / wl - ROPE["low_freq_factor"]) / (ROPE["high_freq_factor"] - ROPE["low_freq_factor"])
    f = torch.where(wl > old / ROPE["low_freq_factor"], f * ROPE["factor"], torch.where(wl > old / ROPE["high_freq_factor"], f / ((1 - s) / ROPE["factor"] + s), f)).to(DEV)

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w

    def rope(x):                                                              # [T, heads, D]
        a = torch.arange(x.shape[0], dtype=F64, device=DEV)[:, None] / f
        c, n = a.cos()[:, None], a.sin()[:, None]
        p, q = x[..., : D // 2], x[..., D // 2:]
        return torch.cat([p * c - q * n, p * n + q * c], -1)

    lens, layer, hs, head, last_norm = [len(r) for r in rows], {}, None, None, None
    for name, t in lm_weights(seed, bits):
        w = _dequantised(t)
        if name == "model.embed_tokens.weight":
            hs = w[torch.from_numpy(np.concatenate(rows).astype(np.int64)).to(DEV)].to(F64)
        elif name == "lm_head.weight":
            head = w
        elif name == "model.norm.weight":
            last_norm = w.to(F64)
        else:
            layer[name.split(".", 3)[3]] = w.to(F64)
        if len(layer) < 9:
            continue
        x = norm(hs, layer["input_layernorm.weight"])
        q, k, v = (x @ layer["self_attn.%s_proj.weight" % n].t() for n in "qkv")
        out, at = [], 0
        for n in lens:
            qq, kk, vv = (y[at: at + n].reshape(n, -1, D) for y in (q, k, v))
            qq, kk = rope(qq).transpose(0, 1), rope(kk).transpose(0, 1).repeat_interleave(H // K, 0)
            vv = vv.transpose(0, 1).repeat_interleave(H // K, 0)
            sc = torch.matmul(qq.contiguous(), kk.transpose(1, 2).contiguous()) / math.sqrt(D)
            sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
            out.append(torch.matmul(sc.softmax(-1), vv.contiguous()).transpose(0, 1).reshape(n, H * D))
            at += n
        hs = hs + torch.cat(out) @ layer["self_attn.o_proj.weight"].t()
        x = norm(hs, layer["post_attention_layernorm.weight"])
        hs = hs + (torch.nn.functional.silu(x @ layer["mlp.gate_proj.weight"].t()) * (x @ layer["mlp.up_proj.weight"].t())) @ layer["mlp.down_proj.weight"].t()
        layer = {}
    last = torch.tensor(np.cumsum(lens) - 1, device=DEV)
    return norm(hs[last], last_norm) @ head.to(F64).t()


class Whisper64:
    def __init__(self, size, seed):
        self.cf = SIZES[size]
        self.w = dict(whisper_weights(size, seed))

    def lin(self, p, x):
        y = x @ self.w[p + ".weight"].to(F64).t()
        return y + self.w[p + ".bias"].to(F64) if p + ".bias" in self.w else y

    def norm(self, p, x):
        return torch.nn.functional.layer_norm(x, (x.shape[-1],), self.w[p + ".weight"].to(F64), self.w[p + ".bias"].to(F64), 1e-5)

    def attend(self, q, k, v):
        """[B, Tq, d], [B, Tk, d]"""
        B, Tq, d = q.shape
        H = self.cf["encoder_attention_heads"]
        q, k, v = (y.reshape(B, -1, H, d // H).transpose(1, 2).contiguous() for y in (q, k, v))
        s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(d // H)
        return torch.matmul(s.softmax(-1), v).transpose(1, 2).reshape(B, Tq, d)

    def encode(self, feats):
        gelu, e = torch.nn.functional.gelu, "model.encoder"
        x = feats.to(F64).transpose(1, 2)
        for n, s in (("conv1", 1), ("conv2", 2)):
            x = gelu(conv(x, self.w["%s.%s.weight" % (e, n)].to(F64).permute(0, 2, 1), self.w["%s.%s.bias" % (e, n)].to(F64), stride=s, pad=1))
        x = x.transpose(1, 2) + self.w[e + ".embed_positions.weight"].to(F64)
        for li in range(self.cf["encoder_layers"]):
            p = "%s.layers.%d" % (e, li)
            h = self.norm(p + ".self_attn_layer_norm", x)
            x = x + self.lin(p + ".self_attn.out_proj", self.attend(*(self.lin("%s.self_attn.%s_proj" % (p, n), h) for n in "qkv")))
            x = x + self.lin(p + ".fc2", gelu(self.lin(p + ".fc1", self.norm(p + ".final_layer_norm", x))))
        return self.norm(e + ".layer_norm", x)

    def first_logits(self, enc):
        """The decoder's logits behind START at position 0 (alone, self-attention returns its own value)."""
        e = "model.decoder"
        x = (self.w[e + ".embed_tokens.weight"][START].to(F64) + self.w[e + ".embed_positions.weight"][0].to(F64)).expand(enc.shape[0], 1, -1)
        for li in range(self.cf["decoder_layers"]):
            p = "%s.layers.%d" % (e, li)
            x = x + self.lin(p + ".self_attn.out_proj", self.lin(p + ".self_attn.v_proj", self.norm(p + ".self_attn_layer_norm", x)))
            h = self.norm(p + ".encoder_attn_layer_norm", x)
            x = x + self.lin(p + ".encoder_attn.out_proj", self.attend(self.lin(p + ".encoder_attn.q_proj", h), self.lin(p + ".encoder_attn.k_proj", enc),
                                                                       self.lin(p + ".encoder_attn.v_proj", enc)))
            x = x + self.lin(p + ".fc2", torch.nn.functional.gelu(self.lin(p + ".fc1", self.norm(p + ".final_layer_norm", x))))
        return self.norm(e + ".layer_norm", x)[:, 0] @ self.w[e + ".embed_tokens.weight"].to(F64).t()


def exact(case, seed):
    k = case["kind"]
    if k == "snac_decode":
        return snac_decode64(snac_weights(seed, False), snac_codes(seed, case["rows"], case["groups"]), seed)
    if k == "snac_encode":
        codes, z = snac_encode64(snac_weights(seed, True), Make(seed, 8).speech(case["rows"], case["samples"], 24000.0))
        return dict(codes=[c.to(torch.int32) for c in codes], z=z)
    if k == "dac_decode":
        cf = dac_config()
        return dac_decode64(dac_weights(seed), Make(seed, 9).ints(0, cf.codebook_size, (case["rows"], cf.n_codebooks, case["frames"])))
    if k == "whisper_encode":
        return Whisper64(case["size"], seed).encode(encoder_features(case, seed))
    if k == "transcribe":
        m, n_mels = Whisper64(case["size"], seed), SIZES[case["size"]]["num_mel_bins"]
        enc = m.encode(torch.stack([log_mel(w, n_mels) for w in windows(case, seed)]))
        says = spoken(seed, 448)[len(PROMPT) - 1: len(PROMPT) - 1 + case["tokens"]]
        return dict(tokens=np.tile(says.astype(np.int32), (case["rows"], 1)), logits=m.first_logits(enc))
    if k == "tts":
        pi, rows, tokens = following(seed), prompts(seed, case["rows"], case["prompt"]), []
        for r in rows:
            t = [int(r[-1])]
            for _ in range(7 * case["frames"]):
                t.append(int(pi[t[-1] - SPEECH0]))
            tokens.append(t[1:])
        tokens = np.asarray(tokens, np.int32)
        logits = lm_logits64(seed, case["bits"], [np.concatenate([r, t, [END_OF_SPEECH]]) for r, t in zip(rows, tokens)])
        spoken_codes = np.concatenate([np.stack([r[-7:] for r in rows]), tokens], 1) - SPEECH0
        c = (spoken_codes.reshape(case["rows"], -1, 7) - np.arange(7) * SLOT).astype(np.int64)
        levels = [c[:, :, [0]], c[:, :, [1, 4]], c[:, :, [2, 3, 5, 6]]]
        levels = [torch.from_numpy(np.ascontiguousarray(v.reshape(case["rows"], -1))).to(DEV) for v in levels]
        return dict(pcm=snac_decode64(snac_weights(seed, False), levels, seed)[:, 0], tokens=tokens, logits=logits)
    return lm_logits64(seed, 0, cloning_prompts(seed, case["rows"], case["prompt"]))
