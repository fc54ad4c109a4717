"""Coefficient offsets of sweeps: 32 bits of bytes from a phase's first
coefficient, so they must not grow with the program or with the circuits that
a batch puts into one table, and a phase with many coefficients is cut (into
parts that hold the same amplitudes in the same registers)."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

CUT = 1 << 16   # coefficients before another phase begins (kMaxPhaseCoefs)
TOL = 1e-10     # 5000 gates x 2^-53 of a unit state, with two orders to spare
N = 8


def _item(layers, seed):
    """Rotations of qubits 0-3 and controlled phases with qubits 4-7: in tiles
    of the 4 low qubits one phase, whose register tables have 256 coefficients."""
    rng = np.random.default_rng(seed)
    c = W.Circuit()
    for i in range(layers):
        for q in range(4):
            c.add("RY", [q], rng.random() * 6)
        for q in range(4):
            c.add("CU1", [q, 4 + (q + i) % 4], lam=rng.random() * 6)
    gates = c.array()
    slots = np.full((len(gates), 3), -1, dtype=np.int32)
    slots[0, 0] = 0
    return {"n": N, "gates": gates, "param_slots": slots, "n_params": 1, "terms": [(1.0, 0, 1), (0.5, 3, 2)],
            "fwd_tile": 4, "adj_tile": 4}


def _err(a, b):
    return max(np.abs(a[0] - b[0]).max(), np.abs(a[1] - b[1]).max())


def test_offsets_do_not_grow_with_the_batch():
    item = _item(20, 3)
    one, off1 = svmi.batch_coefs([item])
    many, off = svmi.batch_coefs([item] * 64)
    assert many == 64 * one and many > CUT
    assert off == off1 < CUT


def test_long_phases_are_cut_and_run_as_one():
    item = _item(300, 4)
    total, off = svmi.batch_coefs([item])
    assert total > CUT > off
    st = W.random_state(N, seed=N)
    assert _err(svmi.emulate(N, item["gates"], st, tile_qubits=4, low_qubits=4), O.run(N, item["gates"], st)) < TOL
    ev, _ = svmi.emulate_batch([item])
    assert abs(ev[0] - O.expval(N, *O.run(N, item["gates"]), item["terms"])) < TOL


def test_long_backward_phases_are_cut():
    # two-qubit blocks on changing pairs, which no other gate joins: 16 coefficients each
    rng = np.random.default_rng(5)
    c = W.Circuit()
    for i in range(4400):
        a, b = (int(q) for q in rng.permutation(4)[:2])
        c.add(("RXX", "RYY", "CRX", "U3")[i % 4], [a, b][:1 if i % 4 == 3 else 2], *(rng.random(3) * 6))
    gates = c.array()
    slots = np.full((len(gates), 3), -1, dtype=np.int32)
    slots[-2, 0] = 0   # CRX, at the start of the backward program
    slots[0, 0] = 1    # RXX, after its cut
    terms, st = [(1.0, 0, 1), (0.5, 3, 2)], W.random_state(4, seed=4)
    e, grad = svmi.emulate_adjoint(4, gates, terms, slots, 2, st)
    assert abs(e - O.expval(4, *O.run(4, gates, st), terms)) < TOL
    v = []
    for s in (np.pi / 2, -np.pi / 2):   # RXX: the two-term rule
        g = gates.copy()
        g["theta"][0] += s
        v.append(O.expval(4, *O.run(4, g, st), terms))
    assert abs(grad[1] - (v[0] - v[1]) / 2) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [False, True])
def test_cut_phases_on_device(compiled):
    item = _item(300, 6)
    ref = O.run(N, item["gates"])
    with svmi.Engine(N) as e:
        e.set_option(svmi.OPT_TILE_QUBITS, 4)
        e.set_option(svmi.OPT_LOW_QUBITS, 4)
        if compiled:
            e.set_option(svmi.OPT_SPECIALIZE, 1)
        e.upload(item["gates"])
        e.run()
        assert (e.stats()["specialized_sweeps"] > 0) == compiled
        assert _err(e.get_state(), ref) < TOL
    if not compiled:
        ev, _ = svmi.batch_adjoint([item, _item(5, 1)])
        assert abs(ev[0] - O.expval(N, *ref, item["terms"])) < TOL
