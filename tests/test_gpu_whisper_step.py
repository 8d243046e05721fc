"""-m gpu: a Whisper decoder step's layers as one launch (csrc/whisper_step.hip): the bits of the launch chain - token ids, and the logits behind the caches it leaves - over widths, depth,
rows, splits of K, positions past a wave's first tile of keys, rows that end, a launch that runs out of time, two handles at once.  Each test says which way the steps went."""
import threading

import numpy as np
import pytest

import mlx_audio_swift_amd as mas

pytestmark = pytest.mark.gpu
PROMPT = [690, 691, 692, 693]


def model(d, layers, vocab=700):
    cfg = mas.WhisperConfig(vocab_size=vocab, num_mel_bins=80, d_model=d, encoder_layers=1, encoder_attention_heads=d // 64, encoder_ffn_dim=d, decoder_layers=layers,
                            decoder_attention_heads=d // 64, decoder_ffn_dim=4 * d)
    return mas.WhisperModel.synthetic(cfg, seed=11)


def transcribe(m, rows, tokens, eot=699, seed=3):
    rng = np.random.default_rng(seed)
    wins = [(0.1 * rng.standard_normal(16000 * (1 + b))).astype(np.float32) for b in range(rows)]
    return m.transcribe_windows(wins, PROMPT, mas.STTGenerateParameters(max_tokens=tokens, temperature=0.0, seed=5, eot_id=eot, timestamp_begin=695))


def run(m, rows, tokens, eot=699, seed=3):
    return transcribe(m, rows, tokens, eot, seed), m.decoder_forward([5 + b for b in range(rows)])


def launches(m):
    """Steps of the last request that went as one launch; requests of this process that ran out of time."""
    lib = mas._lib.lib()
    return lib.mis_debug_whisper_step_launches(m._h), lib.mis_debug_sampler_failures()


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.isfinite(a[1]).all()


# one tile of columns a block and several; one, two, three and five slabs; the last block of a matrix with fewer tiles; 1280 columns at one row: every compute unit;
# eight rows, a norm on each wave; blocks of all matrices (from 1024 columns or 768 and five rows on): one layer, few rows and many blocks, many rows and few blocks
@pytest.mark.parametrize("d,layers,rows", [(384, 2, 5), (384, 4, 8), (768, 2, 8), (1024, 2, 6), (1280, 1, 4), (1280, 3, 3), (1280, 2, 5), (1280, 3, 8), (128, 2, 1), (384, 4, 1), (384, 2, 3), (512, 2, 4), (768, 2, 2), (768, 3, 3), (1024, 2, 1), (1024, 1, 4), (1280, 2, 1)])
def test_bits_of_the_launch_chain(monkeypatch, d, layers, rows):
    m = model(d, layers)
    monkeypatch.setenv("MIS_WHISPER_STEP", "0")
    chain, (none, late) = run(m, rows, 36), launches(m)
    assert none == 0
    monkeypatch.delenv("MIS_WHISPER_STEP")
    for _ in range(2):
        assert same(run(m, rows, 36), chain) and launches(m) == (36, late)


def test_positions_past_the_first_tiles(monkeypatch):
    for d, rows in ((384, 2), (1280, 4)):
        m = model(d, 2)
        monkeypatch.setenv("MIS_WHISPER_STEP", "0")
        chain, (_, late) = run(m, rows, 330), launches(m)
        monkeypatch.delenv("MIS_WHISPER_STEP")
        assert same(run(m, rows, 330), chain) and launches(m) == (330, late)


@pytest.mark.parametrize("d,more_rows", [(384, (2, 4, 6, 9)), (1280, (2, 5))])    # nine: the launch chain
def test_a_row_alone_and_among_others(d, more_rows):
    m = model(d, 2)
    ids, logits = run(m, 1, 20)
    assert launches(m)[0] == 20
    for rows in more_rows:
        more, lm = run(m, rows, 20)
        assert launches(m)[0] == (20 if rows <= 8 else 0)
        assert more[0] == ids[0] and np.array_equal(lm[0], logits[0])


@pytest.mark.parametrize("d,rows", [(384, 2), (1280, 4)])
def test_a_row_that_ends(monkeypatch, d, rows):
    m = model(d, 2)
    full = run(m, rows, 24)[0]
    ends = [t for t in full[1][6:] if t not in full[0]][:1] or [full[1][6]]
    monkeypatch.setenv("MIS_WHISPER_STEP", "0")
    chain, (_, late) = run(m, rows, 24, eot=ends[0])[0], launches(m)
    monkeypatch.delenv("MIS_WHISPER_STEP")
    assert run(m, rows, 24, eot=ends[0])[0] == chain and chain != full
    steps, after = launches(m)
    assert 0 < steps <= 24 and after == late


@pytest.mark.parametrize("d,rows", [(384, 2), (1280, 4)])
def test_out_of_time_runs_on_the_chain(monkeypatch, d, rows):
    m = model(d, 2)
    want, (steps, late) = run(m, rows, 20), launches(m)
    assert steps == 20
    monkeypatch.setenv("MIS_WHISPER_STEP_US", "0")                         # the first poll in vain ends the launch
    got = run(m, rows, 20)
    monkeypatch.delenv("MIS_WHISPER_STEP_US")
    assert same(got, want) and launches(m) == (0, late + 1)
    for steps in (0, 20):                                                  # the next request stays on the launch chain
        assert same(run(m, rows, 20), want) and launches(m) == (steps, late + 1)


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
    """Where the launch chain has room and the values handed between blocks (1 MiB here) have none, or none is left behind them, a request takes the chain."""
    make, call = lambda: model(1280, 2), lambda m: transcribe(m, 8, 20)
    monkeypatch.setenv("MIS_WHISPER_STEP", "0")
    chain, more = run(make(), 8, 20), least(make, call)
    monkeypatch.delenv("MIS_WHISPER_STEP")
    held = mas._lib.lib().mis_debug_device_limit
    for extra, room in ((0, False), (1 << 19, False), (8 << 20, True)):
        m = make()
        late, steps = launches(m)[1], []
        held(more + extra)
        try:
            for _ in range(2):                                             # (the second one's encoder beside what the first one keeps)
                assert call(m) == chain[0]
                steps.append(launches(m)[0])
            assert steps == [20, 20] if room else 0 in steps
        finally:
            held(-1)
        assert same(run(m, 8, 20), chain) and launches(m) == (20, late)


@pytest.mark.parametrize("d,rows", [(768, 2), (1280, 4)])
def test_two_handles_at_once(d, rows):
    ms, rows = [model(384, 2), model(d, 2)], [2, rows]
    want = [run(m, r, 60) for m, r in zip(ms, rows)]
    late = launches(ms[0])[1]
    assert [launches(m)[0] for m in ms] == [60, 60]
    got = [[], []]
    ts = [threading.Thread(target=lambda i=i: got[i].extend(run(ms[i], rows[i], 60) for _ in range(3))) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(same(g, want[i]) for i in range(2) for g in got[i]) and launches(ms[0])[1] == late        # neither waits for the other's compute units


def test_another_call_beside_a_request():
    """From the first poll behind another handle's call on, the launch chain, and the same tokens."""
    m, other = model(384, 4), model(128, 1)
    window, features = (0.1 * np.random.default_rng(3).standard_normal(16000)).astype(np.float32), np.zeros((1, 3000, 80), np.float32)
    gp = mas.STTGenerateParameters(max_tokens=400, temperature=0.0, seed=5, eot_id=699, timestamp_begin=695)
    other.encode(features)
    want = m.transcribe_windows([window], PROMPT, gp)[0]
    steps, late = launches(m)
    assert steps >= len(want) > 300
    got = []
    for e in m.transcribe_windows_stream([window], PROMPT, gp):
        if hasattr(e, "token"):
            got.append(e.token)
            if len(got) == 1:
                other.encode(features)
    here = launches(m)
    assert got == list(want) and 0 < here[0] < steps and here[1] == late
