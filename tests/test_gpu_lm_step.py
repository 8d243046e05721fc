"""-m gpu: the layers of a decode step as one launch (csrc/lm_step.hip): the bits of the launch chain - tokens, samples, and the logits behind the caches it leaves - over depth,
rows, contexts at the edges of key tiles and of the chain's waves, a row that has ended, a launch that runs out of time, two handles at once.  Each test says which way the steps went."""
import threading

import numpy as np
import pytest

import mlx_audio_swift_amd as mas
from mlx_audio_swift_amd.synthetic import snac_synthetic_weights

pytestmark = pytest.mark.gpu

SMALL = dict(encoder_dim=4, encoder_rates=[2, 4, 8, 8], decoder_dim=64, decoder_rates=[8, 8, 4, 2], codebook_size=4096, codebook_dim=8, vq_strides=[4, 2, 1])


def model(layers, **kw):
    cfg = mas.SNACConfig(**SMALL)
    codec = mas.SNAC.from_weights(cfg, snac_synthetic_weights(cfg, seed=1))
    lm = mas.LlamaTTSModel(mas.LlamaTTSConfiguration(hidden_size=3072, num_hidden_layers=layers, intermediate_size=8192, num_attention_heads=24, num_key_value_heads=8, head_dim=128,
                                                     vocab_size=156940, rms_norm_eps=1e-5, rope_theta=500000.0, **kw), codec)
    mas.generation.check(mas._lib.lib().mis_tts_init_synthetic(lm._h, 7))
    lm.finalize()
    return lm


def prompts(rows, n):
    r = np.random.default_rng(3)
    return [np.concatenate([[128259], r.integers(0, 128000, n - 4 - 3 * b), [128009, 128260, 128257]]).astype(np.int32) for b in range(rows)]


def generate(lm, rows, n, tokens):
    pcm, tok = lm.generate_batch(prompts(rows, n), mas.GenerateParameters(max_tokens=tokens, seed=5, temperature=0.8, frame_constrained=2), return_tokens=True)
    return [np.concatenate(pcm), np.concatenate(tok)]


def run(lm, rows, n, tokens):
    return generate(lm, rows, n, tokens) + [lm.lm_forward([128258] * rows)]


def launches(lm):
    """Steps of the last request that went as one launch; requests of this process that ran out of time."""
    lib = mas._lib.lib()
    return lib.mis_debug_tts_step_launches(lm._h), lib.mis_debug_sampler_failures()


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b)) and np.isfinite(a[2]).all()


@pytest.fixture(scope="module")
def three():
    return model(3)


# positions 26 .. 46, 245 .. 265 and 1018 .. 1038: into the second key tile, past the eight waves' first tiles, past k_attn_decode2's caches
@pytest.mark.parametrize("rows,n", [(1, 26), (2, 26), (1, 245), (2, 245), (1, 1018)])
def test_bits_of_the_launch_chain(monkeypatch, three, rows, n):
    monkeypatch.setenv("MIS_LM_STEP", "0")
    chain, (none, late) = run(three, rows, n, 21), launches(three)
    assert none == 0
    monkeypatch.delenv("MIS_LM_STEP")
    for _ in range(2):
        assert same(run(three, rows, n, 21), chain) and launches(three) == (21, late)


@pytest.mark.parametrize("layers", [1, 2])
def test_depth(monkeypatch, layers):
    lm = model(layers)
    monkeypatch.setenv("MIS_LM_STEP", "0")
    chain, (_, late) = run(lm, 2, 40, 70), launches(lm)                    # more steps than one poll of the host's
    monkeypatch.delenv("MIS_LM_STEP")
    assert same(run(lm, 2, 40, 70), chain) and launches(lm) == (70, late)


def test_a_row_alone_and_among_others(three):
    """One row (here), two (here) and three (the chain) of the same batch."""
    (a, na), (b, nb), (c, nc) = [(run(three, r, 40, 14), launches(three)[0]) for r in (1, 2, 3)]
    assert (na, nb, nc) == (14, 14, 0)
    assert np.array_equal(a[1], b[1][:14]) and np.array_equal(b[1], c[1][:28]) and np.array_equal(a[2][0], b[2][0]) and np.array_equal(b[2], c[2][:2])


def test_a_row_that_has_ended(monkeypatch):
    lm = model(2)
    gp = mas.GenerateParameters(max_tokens=28, seed=5, temperature=0.8, frame_constrained=2)
    tok = lm.generate_batch(prompts(2, 40), gp, return_tokens=True)[1]
    ends = [int(t) for t in tok[1][9:12] if t not in tok[0]][0]             # row 1 ends early, row 0 goes on
    lm = model(2, end_of_speech_id=ends)
    monkeypatch.setenv("MIS_LM_STEP", "0")
    chain = lm.generate_batch(prompts(2, 40), gp, return_tokens=True)
    monkeypatch.delenv("MIS_LM_STEP")
    late = launches(lm)[1]
    here = lm.generate_batch(prompts(2, 40), gp, return_tokens=True)
    assert launches(lm) == (28, late) and len(chain[1][1]) < len(chain[1][0])
    assert all(np.array_equal(x, y) for i in range(2) for x, y in zip(chain[i], here[i]))


def test_out_of_time_runs_on_the_chain(monkeypatch):
    """No time to wait at all: the first poll in vain ends every launch, the request runs again on the launch chain; the next request stays there, two after a second time-out in a row."""
    lm = model(2)
    monkeypatch.setenv("MIS_LM_STEP", "0")
    chain, (_, late) = run(lm, 1, 40, 14), launches(lm)
    monkeypatch.delenv("MIS_LM_STEP")
    monkeypatch.setenv("MIS_LM_STEP_US", "0")
    assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (0, late + 1)
    monkeypatch.delenv("MIS_LM_STEP_US")
    assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (0, late + 1)
    monkeypatch.setenv("MIS_LM_STEP_US", "0")
    assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (0, late + 2)
    monkeypatch.delenv("MIS_LM_STEP_US")
    for steps in (0, 0, 14, 14):
        assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (steps, late + 2)
    monkeypatch.setenv("MIS_LM_STEP_US", "0")                              # it got through in between: one request again
    assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (0, late + 3)
    monkeypatch.delenv("MIS_LM_STEP_US")
    for steps in (0, 14):
        assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (steps, late + 3)


def test_a_time_out_of_the_sampler_is_not_the_steps(monkeypatch):
    """A barrier of the one-launch sampler runs out of time: that request runs again, the next one has its steps in one launch."""
    lm = model(2)
    want, (steps, late) = run(lm, 1, 40, 14), launches(lm)
    assert steps == 14
    monkeypatch.setenv("MIS_SAMPLER_SPIN", "0")
    assert same(run(lm, 1, 40, 14), want) and launches(lm) == (0, late + 1)
    monkeypatch.delenv("MIS_SAMPLER_SPIN")
    assert same(run(lm, 1, 40, 14), want) and launches(lm) == (14, late + 1)


def least(make, call):
    """Bytes past a new handle's that two requests of the launch chain get by with, to 64 KiB."""
    held = mas._lib.lib().mis_debug_device_limit
    h = make()
    before = held(-1)
    call(h)
    more = held(-1) - before
    while True:
        h = make()
        held(more)
        try:
            call(h), call(h)
            return more
        except mas.generation.AudioGenerationError:
            more += 1 << 16
        finally:
            held(-1)


def test_no_room_for_the_step(monkeypatch):
    """Where the launch chain has room and the values handed between blocks (180 KiB here) have none, or none is left behind them, a request takes the chain."""
    make, call = lambda: model(2), lambda lm: generate(lm, 1, 40, 14)
    monkeypatch.setenv("MIS_LM_STEP", "0")
    chain, more = run(make(), 1, 40, 14), least(make, call)
    monkeypatch.delenv("MIS_LM_STEP")
    held = mas._lib.lib().mis_debug_device_limit
    for extra, steps in ((0, 0), (100 << 10, 0), (1 << 20, 14)):
        lm = make()
        late = launches(lm)[1]
        held(more + extra)
        try:
            for _ in range(2):
                got = call(lm)
                assert launches(lm)[0] == steps
                assert all(np.array_equal(x, y) for x, y in zip(got, chain))
        finally:
            held(-1)
        assert same(run(lm, 1, 40, 14), chain) and launches(lm) == (14, late)


def test_two_handles_at_once(three):
    other = model(3)
    want, (steps, late) = run(three, 1, 40, 70), launches(three)
    assert steps == 70
    got = {}

    def work(name, lm):
        got[name] = [run(lm, 1, 40, 70) for _ in range(3)]
    threads = [threading.Thread(target=work, args=(k, m)) for k, m in (("a", three), ("b", other))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(same(r, want) for k in "ab" for r in got[k]) and launches(three)[1] == late        # neither waits for the other's compute units


@pytest.mark.parametrize("graph", [True, False])                          # the handle has a graph of the chain's steps, or none yet
@pytest.mark.parametrize("other", ["codec", "sampler"])                   # the sampler's blocks wait for each other, its copies go over the legacy stream
def test_another_call_beside_a_request(monkeypatch, three, graph, other):
    """From the first poll behind another handle's call on, the launch chain, and the same tokens."""
    cfg = mas.SNACConfig(**SMALL)
    codec = mas.SNAC.from_weights(cfg, snac_synthetic_weights(cfg, seed=1))
    codes, logits = [np.zeros((1, k), np.int32) for k in (1, 2, 4)], np.random.default_rng(0).standard_normal((8, 30000)).astype(np.float32)
    calls = dict(codec=lambda: codec.decode(codes),
                 sampler=lambda: mas.tts.sample_logits(logits, np.zeros((8, 0), np.int32), np.zeros(8, np.int32), mas.GenerateParameters(temperature=0.8, top_p=0.9), 0))
    calls[other]()
    gp = mas.GenerateParameters(max_tokens=600, seed=5, temperature=0.8, frame_constrained=2)
    if not graph:
        three.generate_batch(prompts(1, 41), gp)                           # (another prompt length: the graphs of the one before go)
    else:
        monkeypatch.setenv("MIS_LM_STEP", "0")
        for _ in three.generate_stream_batch(prompts(1, 40), gp):
            pass
        monkeypatch.delenv("MIS_LM_STEP")
    want = three.generate_batch(prompts(1, 40), gp, return_tokens=True)[1][0]
    steps, late = launches(three)
    assert steps >= len(want) > 500
    got = []
    for e in three.generate_stream_batch(prompts(1, 40), gp):
        if hasattr(e, "token"):
            got.append(e.token)
            if len(got) == 1:
                calls[other]()
    here = launches(three)
    assert np.array_equal(got, want) and 0 < here[0] < steps and here[1] == late
