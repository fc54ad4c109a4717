"""Pauli sums evaluated tile by tile: masks inside a tile, across two tiles'
qubits, and masks no tile holds, with real and imaginary coefficients (odd
numbers of Y) -- on the CPU through the adjoint emulation, whose 6-qubit tiles
give small states several passes, and on the GPU at the sizes where the tile
(8, 10, 12 qubits) and the number of passes change."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

# sums of 2^n products with |coefficients| ~ 1 and a unit state: the error of
# either side is far below n_terms * 2^-50
TOL = 1e-12


def _terms(n, rng, count):
    full = (1 << n) - 1
    t = [(float(c), x, z) for c, x, z in W.ising_terms(n, rng)] if n > 1 else [(0.7, 1, 0)]
    for _ in range(count):
        x = int(rng.integers(0, 1 << n)) & int(rng.integers(0, 1 << n)) & full   # about a quarter of the qubits
        t.append((float(rng.standard_normal()), x, int(rng.integers(0, 1 << n))))
    t += [(0.5, full, full), (0.25, full, 0), (-0.75, 1 << (n - 1), 1 << (n - 1))]
    return t


@pytest.mark.parametrize("n", [4, 6, 7, 9, 11])
def test_emulated_passes_match_oracle(n):
    rng = np.random.default_rng(40 + n)
    st = W.random_state(n, seed=n)
    gates = svmi.as_gates([("RY", (q,), 0.1 * (q + 1)) for q in range(n)])
    slots = np.full((n, 3), -1, dtype=np.int32)
    slots[:, 0] = np.arange(n)
    for terms in (_terms(n, rng, 12), [(float(c), x, z) for c, x, z in W.ising_terms(n, rng)]):
        e, grad = svmi.emulate_adjoint(n, gates, terms, slots, n, st)
        assert abs(e - O.expval(n, *O.run(n, gates, st), terms)) < TOL * len(terms)
        for q in (0, n - 1):   # lambda = H psi went through the same passes
            v = []
            for s in (np.pi / 2, -np.pi / 2):
                g = gates.copy()
                g["theta"][q] += s
                v.append(O.expval(n, *O.run(n, g, st), terms))
            assert abs(grad[q] - (v[0] - v[1]) / 2) < TOL * len(terms)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 12, 17, 18, 19, 20, 22, 23])
def test_expval_on_device_matches_oracle(n):
    rng = np.random.default_rng(60 + n)
    st = W.random_state(n, seed=n)
    ising = [(float(c), x, z) for c, x, z in W.ising_terms(n, rng)] if n > 1 else [(0.7, 1, 0)]
    with svmi.Engine(n) as e:
        e.set_state(*st)
        for terms in (ising, _terms(n, rng, 6), [(0.3, 0, 0)], [(1.5, 1 << (n - 1), 0)], []):
            assert abs(e.expval(terms) - O.expval(n, *st, terms)) < TOL * max(len(terms), 1)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5, 13, 18, 22])
def test_adjoint_lambda_through_passes(n):
    rng = np.random.default_rng(80 + n)
    gates, slots, p = W.hea(n, 1, rng)
    terms = _terms(n, rng, 3)
    with svmi.Engine(n) as e:
        e.upload(gates)
        E, grad = e.adjoint(terms, slots, p)
    ev, gr = svmi.batch_adjoint([{"n": n, "gates": gates, "param_slots": slots, "n_params": p, "terms": terms}])
    ore = O.run(n, gates)
    assert abs(E - O.expval(n, *ore, terms)) < TOL * len(terms) and abs(ev[0] - E) < TOL * len(terms)
    assert np.abs(grad - gr[0]).max() < TOL * len(terms)
    for q in (0, n - 1):
        v = []
        for s in (np.pi / 2, -np.pi / 2):
            g = gates.copy()
            g["theta"][q] += s
            v.append(O.expval(n, *O.run(n, g), terms))
        assert abs(grad[q] - (v[0] - v[1]) / 2) < TOL * len(terms)
