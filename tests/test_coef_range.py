"""Coefficient offsets of sweeps: 32 bits of bytes from a sweep's first
coefficient, so they must not grow with the sweeps of a program or with the
circuits that a batch puts into one table."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

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
    assert many == 64 * one and off == off1 < one


def test_offsets_do_not_grow_with_the_sweeps():
    # brick walls over more qubits than a tile has: sweeps of like size follow each other
    def item(layers):
        gates = W.u3_brickwall(16, layers)
        return {"n": 16, "gates": gates, "param_slots": np.full((len(gates), 3), -1, dtype=np.int32), "n_params": 0,
                "terms": [(1.0, 0, 1)], "fwd_tile": 8, "adj_tile": 8}
    few, off_few = svmi.batch_coefs([item(6)])
    many, off = svmi.batch_coefs([item(24)])
    assert many > 3 * few and off < 2 * off_few


def test_large_tables_match_oracle():
    item = _item(300, 4)
    total, off = svmi.batch_coefs([item])
    assert total > 1 << 16
    st = W.random_state(N, seed=N)
    assert _err(svmi.emulate(N, item["gates"], st, tile_qubits=4, low_qubits=4), O.run(N, item["gates"], st)) < TOL
    ev, _ = svmi.emulate_batch([item])
    assert abs(ev[0] - O.expval(N, *O.run(N, item["gates"]), item["terms"])) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [False, True])
def test_large_tables_on_device(compiled):
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
        ev, _ = svmi.batch_adjoint([_item(5, 1), item])
        assert abs(ev[1] - O.expval(N, *ref, item["terms"])) < TOL
