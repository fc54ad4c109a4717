"""Register layouts of sweeps: the exchanges between phases, loads and stores.

On the CPU the program runs as the device does it -- register groups per
thread, exchanges through slots, waves checked where no barrier is planned --
at tile sizes from one thread to 512, at every number of low qubits, with
and without tile maps.  On the GPU the sizes where the kernel changes (few
tiles: latency build; blocks of three and four qubits), and sweeps that only
relabel, whose waves store where others load, twice with the same bits."""
import numpy as np
import pytest

import svmi
from oracle import oracle as O
from svmi import workloads as W

TOL = 1e-12   # depth x 2^-53 of a unit state, with two orders to spare


def _circuit(n, rng, wide):
    g = svmi.workloads.Circuit()
    for _ in range(3):
        for q in range(n):
            g.add(("RX", "RY", "H", "U3")[int(rng.integers(4))], [q], *(rng.random(3) * 6))
        perm = [int(q) for q in rng.permutation(n)]
        for i in range(0, n - 1, 2):
            g.add(("CX", "SWAP", "CZ", "CRY", "CU1")[int(rng.integers(5))], perm[i:i + 2], 0.3, 0.4, 0.5)
        if wide and n >= 4:
            g.add("CCX", perm[:3])
            g.add("RC3X", perm[-4:])
    return g.array()


def _err(a, b):
    return max(np.abs(a[0] - b[0]).max(), np.abs(a[1] - b[1]).max())


@pytest.mark.parametrize("n", [4, 7, 11, 14])
@pytest.mark.parametrize("tile,low", [(13, 3), (13, 6), (12, 2), (11, 4), (10, 0), (7, 3), (5, 4), (4, 4)])
def test_emulated_layouts_match_oracle(n, tile, low):
    rng = np.random.default_rng(1000 * n + 10 * tile + low)
    gates = _circuit(n, rng, wide=True)
    st = W.random_state(n, seed=n)
    assert _err(svmi.emulate(n, gates, st, tile_qubits=tile, low_qubits=low), O.run(n, gates, st)) < TOL
    q = W.qft(n)
    assert _err(svmi.emulate(n, q, st, tile_qubits=tile, low_qubits=low), O.run(n, q, st)) < TOL


@pytest.mark.parametrize("n", [5, 9, 13])
@pytest.mark.parametrize("tile,low", [(12, 3), (11, 4), (8, 2), (6, 0)])
def test_emulated_two_state_layouts_match_oracle(n, tile, low):
    rng = np.random.default_rng(77 * n + tile)
    gates, slots, p = W.hea(n, 2, rng)
    terms = W.ising_terms(n, rng)
    st = W.random_state(n, seed=n)
    e, grad = svmi.emulate_adjoint(n, gates, terms, slots, p, st, tile_qubits=tile, low_qubits=low)
    assert abs(e - O.expval(n, *O.run(n, gates, st), terms)) < TOL * len(terms)
    for k in (0, p - 1):
        v = []
        for s in (np.pi / 2, -np.pi / 2):
            g = gates.copy()
            i, f = np.argwhere(slots == k)[0]
            g[("theta", "phi", "lambda")[f]][i] += s
            v.append(O.expval(n, *O.run(n, g, st), terms))
        # RY: the two-term rule; RZ turns one amplitude only, the same rule up to a global phase
        assert abs(grad[k] - (v[0] - v[1]) / 2) < TOL * len(terms)


@pytest.mark.gpu
@pytest.mark.parametrize("n,tile,low", [(4, 13, 4), (9, 13, 3), (13, 13, 3), (14, 13, 3), (16, 9, 3), (19, 12, 4),
                                        (20, 12, 4), (20, 13, 3), (21, 12, 2), (21, 13, 3)])
def test_device_layouts_match_oracle(n, tile, low):
    rng = np.random.default_rng(31 * n + tile)
    st = W.random_state(n, seed=n)
    for wide in (False, True):
        gates = _circuit(n, rng, wide)
        with svmi.Engine(n) as e:
            e.set_option(svmi.OPT_TILE_QUBITS, tile)
            e.set_option(svmi.OPT_LOW_QUBITS, low)
            e.upload(gates)
            e.set_state(*st)
            e.run()
            got = e.get_state()
        assert _err(got, O.run(n, gates, st)) < TOL, wide


@pytest.mark.gpu
@pytest.mark.parametrize("tile,low", [(12, 4), (13, 4), (13, 3)])
def test_relabelling_sweeps_give_the_same_bits_every_time(tile, low):
    n = 22
    swaps = svmi.workloads.Circuit()
    for i in range(n // 2):
        swaps.add("SWAP", [i, n - 1 - i])
    for i in range(n - 1):
        swaps.add("CX", [i, i + 1])
    st = W.random_state(n, seed=22)
    for gates in (swaps.array(), W.qft(n)):
        with svmi.Engine(n) as e:
            e.set_option(svmi.OPT_TILE_QUBITS, tile)
            e.set_option(svmi.OPT_LOW_QUBITS, low)
            e.upload(gates)
            first = None
            for _ in range(3):
                e.set_state(*st)
                e.run()
                got = e.get_state()
                first = first or got
                assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1])
        assert _err(first, O.run(n, gates, st)) < TOL
