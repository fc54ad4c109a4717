"""How Pauli sums are planned: one pass on the states that the last-level cache
holds, several above where masks share tiles, smaller tiles where hardly any
mask lies in one; planning time linear in the masks.  On the GPU the plans of
smaller tiles against the oracle."""
import time

import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

TOL = 1e-12   # per term: sums of 2^n products of a unit state


def _random_terms(n, count, seed, weight=None):
    """Terms of random masks; weight: of that many qubits at least."""
    rng = np.random.default_rng(seed)
    x = rng.integers(0, 1 << n, size=count)
    if weight is not None:
        x = np.array([sum(1 << int(q) for q in rng.choice(n, size=weight, replace=False)) for _ in range(count)]) | x
    return list(zip(rng.standard_normal(count), x.tolist(), rng.integers(0, 1 << n, size=count).tolist()))


def _ising(n):
    return [(float(c), x, z) for c, x, z in W.ising_terms(n, np.random.default_rng(n))]


@pytest.mark.parametrize("n", [8, 14, 17, 19, 20, 21])
@pytest.mark.parametrize("lam", [False, True])
def test_states_in_the_cache_take_one_pass(n, lam):
    for terms in (_ising(n), _random_terms(n, 50, n)):
        assert svmi.plan_pauli(n, terms, lam)["passes"] == 1


@pytest.mark.parametrize("n", [22, 25, 28, 33])
def test_larger_states_take_passes_and_tiles_by_their_masks(n):
    p = svmi.plan_pauli(n, _ising(n))
    # the 12 lowest qubits, then 8 of the others at a time
    assert p == {"passes": 1 + -(-(n - 12) // 8), "tile_qubits": 12, "in_tile": n + 1, "from_memory": 0}
    terms = _random_terms(n, 30, n, weight=n - 4)
    masks = len({x for _, x, _ in terms})
    assert svmi.plan_pauli(n, terms) == {"passes": 1, "tile_qubits": 10, "in_tile": 0, "from_memory": masks}


def test_planning_is_linear_in_the_masks():
    n = 27   # masks of 20 qubits and more: no two share a tile

    def best(terms):
        t = svmi.as_terms(terms)
        times = []
        for _ in range(3):
            t0 = time.perf_counter()
            svmi.plan_pauli(n, t)
            times.append(time.perf_counter() - t0)
        return min(times)

    terms = _random_terms(n, 40000, 3, weight=20)
    assert best(terms) < 9 * best(terms[:10000])   # 4 if linear, 16 if every mask looks at all others


@pytest.mark.gpu
@pytest.mark.parametrize("n", [20, 22, 23])
def test_memory_bound_sums_match_oracle(n):
    terms = _random_terms(n, 9, n, weight=n - 6) + [(0.5, 1, 1)]
    assert svmi.plan_pauli(n, terms)["tile_qubits"] == svmi.plan_pauli(n, terms, True)["tile_qubits"] == 10
    st = W.random_state(n, seed=n)
    with svmi.Engine(n) as e:
        e.set_state(*st)
        assert abs(e.expval(terms) - O.expval(n, *st, terms)) < TOL * len(terms)
        gates, slots, p = W.hea(n, 1, np.random.default_rng(n))
        e.reset_state()
        e.upload(gates)
        E, grad = e.adjoint(terms, slots, p)
    assert abs(E - O.expval(n, *O.run(n, gates), terms)) < TOL * len(terms)
    ev, gr = svmi.batch_adjoint([{"n": n, "gates": gates, "param_slots": slots, "n_params": p, "terms": terms}])
    assert abs(E - ev[0]) < TOL * len(terms) and np.abs(grad - gr[0]).max() < TOL * len(terms)
