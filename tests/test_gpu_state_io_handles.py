"""GPU: set_state / get_state on new handles: the caller's thread alone (up to 3
runs of 2 chunks of 2^17 amplitudes) and with helpers that take runs as well,
also while other threads keep the cores busy; the slots of the process handed
from one handle to the next.  Copies, so every bit must come back."""
import threading

import numpy as np
import pytest

import svmi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 17, 18, 19, 20, 22])
def test_handles_one_after_another(n):
    rng = np.random.default_rng(n)
    for _ in range(3):
        re, im = rng.standard_normal(1 << n), rng.standard_normal(1 << n)
        with svmi.Engine(n) as e:
            e.set_state(re, im)
            r, i = e.get_state()
            assert np.array_equal(r, re) and np.array_equal(i, im)


def test_handles_side_by_side():
    rng = np.random.default_rng(1)
    states = [(n, rng.standard_normal(1 << n), rng.standard_normal(1 << n)) for n in (3, 19, 20, 18)]
    engines = [svmi.Engine(n) for n, _, _ in states]
    for e, (_, re, im) in zip(engines, states):
        e.set_state(re, im)
    for e, (_, re, im) in reversed(list(zip(engines, states))):
        r, i = e.get_state()
        assert np.array_equal(r, re) and np.array_equal(i, im)
        e.close()


def test_copies_beside_busy_threads():
    # helpers that come late, or in the middle, or not at all
    stop = threading.Event()

    def spin():
        a = np.arange(1 << 16, dtype=np.float64)
        while not stop.is_set():
            np.sin(a, out=a)   # without the interpreter's lock

    threads = [threading.Thread(target=spin) for _ in range(24)]
    for t in threads:
        t.start()
    try:
        rng = np.random.default_rng(2)
        for n in (20, 21, 20):
            re, im = rng.standard_normal(1 << n), rng.standard_normal(1 << n)
            with svmi.Engine(n) as e:
                for _ in range(3):
                    e.set_state(re, im)
                    r, i = e.get_state()
                    assert np.array_equal(r, re) and np.array_equal(i, im)
                    re, im = im, re
    finally:
        stop.set()
        for t in threads:
            t.join()
