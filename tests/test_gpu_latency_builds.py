"""GPU: where sweeps of few tiles change their kernel -- tiles of less than one
wave (whose other lanes repeat them), one wave and eight, from one tile to the
2^17 threads above which the ordinary build runs, exchanges of whole amplitudes
and by halves -- one state and two, against the oracle."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

pytestmark = pytest.mark.gpu
TOL = 1e-12   # depth x 2^-53 of a unit state, with two orders to spare


@pytest.mark.parametrize("n,tile", [(4, 12), (5, 12), (6, 4), (7, 5), (8, 12), (9, 6), (10, 10), (11, 12), (13, 13),
                                    (14, 12), (15, 4), (16, 6), (19, 13), (20, 10), (20, 13), (21, 10), (22, 10)])
def test_small_sweeps_match_oracle(n, tile):
    rng = np.random.default_rng(5 * n + tile)
    st = W.random_state(n, seed=n)
    for gates in (W.random_layers(n=n, layers=4, seed=int(rng.integers(1 << 30))), W.qft(n)):
        with svmi.Engine(n) as e:
            e.set_option(svmi.OPT_TILE_QUBITS, tile)
            e.set_option(svmi.OPT_LOW_QUBITS, 3)
            e.upload(gates)
            e.set_state(*st)
            e.run()
            re, im = e.get_state()
        ore, oim = O.run(n, gates, st)
        assert max(np.abs(re - ore).max(), np.abs(im - oim).max()) < TOL


@pytest.mark.parametrize("n,tile", [(4, 12), (5, 4), (6, 12), (8, 5), (9, 12), (12, 12), (12, 4), (16, 11), (19, 9)])
def test_small_gradients_match_shifted_energies(n, tile):
    rng = np.random.default_rng(9 * n + tile)
    gates, slots, p = W.hea(n, 2, rng)
    terms = [(float(c), x, z) for c, x, z in W.ising_terms(n, rng)]
    with svmi.Engine(n) as e:
        e.set_option(svmi.OPT_TILE_QUBITS, tile)
        e.set_option(svmi.OPT_LOW_QUBITS, 3)
        e.upload(gates)
        E, grad = e.adjoint(terms, slots, p)
    assert abs(E - O.expval(n, *O.run(n, gates), terms)) < TOL * len(terms)
    for k in (0, p - 1) if n > 12 else rng.choice(p, size=4, replace=False):
        i, f = np.argwhere(slots == k)[0]
        v = []
        for s in (np.pi / 2, -np.pi / 2):
            g = gates.copy()
            g[("theta", "phi", "lambda")[f]][i] += s
            v.append(O.expval(n, *O.run(n, g), terms))
        assert abs(grad[k] - (v[0] - v[1]) / 2) < TOL * len(terms)


@pytest.mark.parametrize("count,n,kw", [(1, 4, {}), (3, 5, {}), (3, 7, {"fwd_tile": 6, "adj_tile": 6}), (2, 9, {}),
                                        (4, 12, {}), (300, 4, {}), (6, 12, {"fwd_tile": 6, "adj_tile": 7}),
                                        (2, 15, {}), (3, 17, {"fwd_tile": 12, "adj_tile": 11})])
def test_small_batches_match_single_circuits(count, n, kw):
    rng = np.random.default_rng(count + 100 * n)
    items = []
    for i in range(count):
        gates, slots, p = W.hea(n, 1 + i % 3, rng)
        terms = [(float(c), x, z) for c, x, z in W.ising_terms(n, rng)]
        items.append(dict({"n": n, "gates": gates, "param_slots": slots, "n_params": p, "terms": terms}, **kw))
    ev, grads = svmi.batch_adjoint(items)
    for i, it in enumerate(items):
        tol = TOL * len(it["terms"])
        assert abs(ev[i] - O.expval(n, *O.run(n, it["gates"]), it["terms"])) < tol
        if i < 4:
            with svmi.Engine(n) as e:
                e.upload(it["gates"])
                _, g = e.adjoint(it["terms"], it["param_slots"], it["n_params"])
            assert np.abs(g - grads[i]).max() < tol
