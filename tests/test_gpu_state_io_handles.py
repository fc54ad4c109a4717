"""GPU: set_state / get_state on new handles: the caller's thread cycling
through the slots, from 32 chunks of 2^17 amplitudes on four workers with a
quarter each, the slots of the process handed from one handle to the next.  Copies, so every
bit must come back."""
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
