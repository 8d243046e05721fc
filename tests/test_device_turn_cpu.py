"""Which request may have its decode steps in one launch (DeviceCall, DeviceTurn, device_settle: csrc/common.h): one that is alone on its device.  Threads in turn, no device."""
import queue
import threading
import time

import pytest

from mlx_audio_swift_amd import _lib

ENTER, LEAVE, TAKE, REST, POLL, GIVE, SETTLE = range(7)
QUIET, SETTLE_S = 0.05, 0.5
DEVICES = iter(range(8, 60))                                               # a test's own


class Caller:
    """A thread that does one thing after the other for the test."""

    def __init__(self, device):
        self.device, self.todo, self.done = device, queue.Queue(), queue.Queue()
        self.thread = threading.Thread(target=self._run, daemon=True)
        self.thread.start()

    def _run(self):
        for op in iter(self.todo.get, None):
            self.done.put(_lib.lib().mis_debug_device_turn(self.device, op))

    def begin(self, op):
        self.todo.put(op)

    def end(self, timeout=5):
        return self.done.get(timeout=timeout)

    def __call__(self, op):
        self.begin(op)
        return self.end()


@pytest.fixture
def two():
    device = next(DEVICES)
    both = Caller(device), Caller(device)
    yield both
    for c in both:
        c.todo.put(None)
        c.thread.join()


def test_alone_until_another_call_comes(two):
    a, b = two
    a(ENTER)
    assert a(TAKE) == 1 and a(POLL) == 1
    b(ENTER)
    assert b(TAKE) == 0
    assert a(POLL) == 0 and b(POLL) == 0                                   # neither, beside each other
    t = time.perf_counter()
    assert a(POLL) == 0
    b(LEAVE)
    assert a(POLL) == 0 or time.perf_counter() - t >= QUIET
    time.sleep(QUIET + 0.02)
    assert a(POLL) == 1                                                    # alone for a while
    a(GIVE), a(LEAVE)
    b(ENTER)
    assert b(TAKE) == 1
    b(GIVE), b(LEAVE)


def test_a_call_that_has_gone_again(two):
    """A call between two polls counts, and each one begins the wait anew."""
    a, b = two
    a(ENTER)
    assert a(TAKE) == 1
    for _ in range(3):
        b(ENTER), b(LEAVE)
        t = time.perf_counter()
        assert a(POLL) == 0
        time.sleep(0.6 * QUIET)
    assert a(POLL) == 0 or time.perf_counter() - t >= QUIET
    time.sleep(QUIET)
    assert a(POLL) == 1
    a(GIVE), a(LEAVE)


def test_calls_inside_a_call_are_part_of_it(two):
    a, b = two
    a(ENTER)
    assert a(TAKE) == 1
    a(REST), a(ENTER), a(SETTLE), a(LEAVE)                                 # an event callback's: no wait for itself
    assert a(POLL) == 1
    b(ENTER)
    assert a(POLL) == 0
    b(LEAVE), a(LEAVE)


def test_kernels_whose_blocks_wait(two):
    """Until the request that has the device has polled; not while it rests; bounded."""
    a, b = two
    a(ENTER), a(TAKE), b(ENTER)
    b.begin(SETTLE)
    with pytest.raises(queue.Empty):
        b.end(0.1)
    assert a(POLL) == 0
    b.end(0.4)
    b(LEAVE), a(GIVE), a(LEAVE)
    a(ENTER)
    assert a(TAKE) == 1
    a(REST), b(ENTER)
    t = time.perf_counter()
    b(SETTLE)
    assert time.perf_counter() - t < 0.6 * SETTLE_S and a(POLL) == 0
    b(LEAVE), a(LEAVE)
    a(ENTER)
    assert a(TAKE) == 1
    b(ENTER)
    t = time.perf_counter()
    b(SETTLE)
    assert 0.9 * SETTLE_S < time.perf_counter() - t < 4 * SETTLE_S
    b(LEAVE), a(GIVE), a(LEAVE)


def test_no_call_no_turn_and_devices_past_the_table(two):
    a, _ = two
    assert a(TAKE) == 0
    lib = _lib.lib()
    assert [lib.mis_debug_device_turn(1000, op) for op in (ENTER, TAKE, POLL, SETTLE, GIVE, LEAVE)] == [0] * 6
    assert [lib.mis_debug_device_turn(-1, op) for op in (ENTER, TAKE, POLL, SETTLE, GIVE, LEAVE)] == [0] * 6
