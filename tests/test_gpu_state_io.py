"""GPU: set_state / get_state through the pinned slots: sizes of less than one
slot (2^17 amplitudes), one, two, one per worker and several per worker, and
two handles at once from two threads.  Copies, so every bit must come back."""
import threading

import numpy as np
import pytest

import svmi

pytestmark = pytest.mark.gpu


def _round_trip(n, seed):
    rng = np.random.default_rng(seed)
    re, im = rng.standard_normal(1 << n), rng.standard_normal(1 << n)
    with svmi.Engine(n) as e:
        for _ in range(2):
            e.set_state(re, im)
            idx = rng.integers(0, 1 << n, size=64).astype(np.uint64)
            a, b = e.get_amplitudes(idx)
            assert np.array_equal(a, re[idx]) and np.array_equal(b, im[idx])
            r, i = e.get_state()
            assert np.array_equal(r, re) and np.array_equal(i, im)
            re, im = im, re


@pytest.mark.parametrize("n", [1, 4, 16, 17, 18, 19, 21])
def test_state_round_trip(n):
    _round_trip(n, n)


def test_state_round_trip_from_two_threads():
    failed = []

    def work(seed):
        try:
            _round_trip(19, seed)
        except Exception as e:   # noqa: BLE001 -- reported below
            failed.append(e)

    t = [threading.Thread(target=work, args=(s,)) for s in (1, 2, 3)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not failed
