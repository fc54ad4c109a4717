"""GPU: sampling against the oracle's scan, draw for draw.  The states hold
probabilities of 2^-2m on a random subset of the basis states, so every
partial sum is exact in any order and even a draw that lies on an interval's
end has one right answer; runs of zeros test the ties."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,shots", [(2, 1, 5), (4, 1, 300), (6, 2, 64), (9, 3, 257), (12, 0, 256), (12, 5, 1024),
                                       (13, 5, 4097), (16, 6, 5000), (17, 4, 3)])
def test_samples_equal_oracle_on_exact_probabilities(n, m, shots):
    rng = np.random.default_rng(100 * n + m)
    re, im = np.zeros(1 << n), np.zeros(1 << n)
    at = np.sort(rng.choice(1 << n, size=4 ** m, replace=False))
    part = rng.integers(2, size=4 ** m)
    sign = rng.choice([-1.0, 1.0], size=4 ** m)
    re[at] = np.where(part == 0, sign * 2.0 ** -m, 0.0)
    im[at] = np.where(part == 1, sign * 2.0 ** -m, 0.0)
    u = rng.random(shots)
    edge = rng.integers(0, 4 ** m + 1, size=shots) / 4 ** m   # interval ends, 0 and 1 among them
    u[::2] = edge[::2]
    with svmi.Engine(n) as e:
        e.set_state(re, im)
        got, total = e.measure(u)
    assert total == 1.0
    assert np.array_equal(got, O.measure(n, re, im, u))
