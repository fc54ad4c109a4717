"""Compiled sweeps on the register layouts, where addresses can go wrong:
tiles of less than a wave up to several waves, sweeps that only move
amplitudes (with and without tile maps: below and from 20 qubits on), 13-qubit
tiles (from 20 qubits on), and
phase products read from the staged lane tables.

Permutation circuits only move numbers, so their states equal the oracle's
exactly.  The phase circuits multiply each amplitude by at most 12 n rounded
factors, each good to a few 2^-53 relative, on a state of unit norm: 1e-12.
"""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

pytestmark = pytest.mark.gpu


def _run(n, gates, state, tile=None, low=None):
    with svmi.Engine(n) as e:
        e.set_option(svmi.OPT_SPECIALIZE, 1)
        if tile is not None:
            e.set_option(svmi.OPT_TILE_QUBITS, tile)
        if low is not None:
            e.set_option(svmi.OPT_LOW_QUBITS, low)
        e.set_state(*state)
        e.upload(gates)
        e.run()
        assert e.stats()["specialized_sweeps"] > 0
        return e.get_state()


CASES = [(5, None, None), (9, None, None), (10, None, None), (11, None, None), (13, None, None), (13, 5, 0),
         (14, 9, 3), (19, None, None), (20, None, None), (20, 13, 3), (20, 12, 3)]


@pytest.mark.parametrize("n,tile,low", CASES)
def test_permutations_are_exact(n, tile, low):
    print(f"case: n={n} tile={tile} low={low}", flush=True)
    rng = np.random.default_rng(700 + n)
    X, CX, SWAP = (svmi.OP_NAMES.index(s) for s in ("X", "CX", "SWAP"))
    gates = []
    for _ in range(60):
        a, b = (int(v) for v in rng.choice(n, size=2, replace=False))
        gates.append(((X, [a]), (CX, [a, b]), (SWAP, [a, b]))[int(rng.integers(3))] + (0.0, 0.0, 0.0))
    st = W.random_state(n, seed=n)
    got = _run(n, gates, st, tile, low)
    want = O.run(n, gates, st)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("n,tile,low", CASES)
def test_phase_products(n, tile, low):
    print(f"case: n={n} tile={tile} low={low}", flush=True)
    gates = W.qft(n=n)
    st = W.random_state(n, seed=n + 1)
    got = _run(n, gates, st, tile, low)
    want = O.run(n, gates, st)
    assert max(np.abs(got[0] - want[0]).max(), np.abs(got[1] - want[1]).max()) < 1e-12
