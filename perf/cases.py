"""Performance cases of the state-vector engine: what a program that uses it
has it do, through the public entry points of the svmi package, and what the
same call gives in plain torch (complex128) without it.

A case is a dict with a "kind":

  shots    layers of random {H, RX, RY, RZ} + CX pairs from |0..0>, sampled and
           read back whole: the everyday small circuit, bound by latency.
  job      one OpenQASM 2.0 circuit from its text to its samples and its state:
           parse, upload (lowering and scheduling on the host), run, measure.
           A service that is handed one circuit after another.
  state    a program that keeps its own copy of the state: set_state, a circuit,
           get_state (the reference's public sv_real / sv_imag members).
  xeb      U3 brick wall from |0..0>, samples drawn and the amplitudes of given
           bitstrings read: random circuit sampling with its cross-entropy check.
  qft      quantum Fourier transform of the state that is there, then samples and
           amplitudes: phase-heavy circuits.  "compiled" turns on
           OPT_SPECIALIZE, for circuits that run many times.
  qir      a QIR gate-set program with multi-controlled gates and mid-circuit
           measurements, planned on each call as the QIR driver does.
  dm       the same program on a density matrix of n qubits (2n-qubit state).
  energy   <H> of an Ising Hamiltonian on a state that is there.
  train    one step of gradient descent on <H> of a hardware-efficient ansatz
           through torch.autograd: new angles are bound, uploaded and
           differentiated on every step.
  grad     the adjoint gradient of a circuit that stays uploaded.
  batch    the gradients of many uneven circuits in one call.

Whole states come back where a program would read them (up to some 20 qubits);
from larger ones a program reads samples and the amplitudes of the bitstrings
that it is asked about, and these are returned as read.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "sv-sim_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_RAND_MAX = 2147483647
_AMPS = 16384   # bitstrings whose amplitudes are read from a large state


def listed():
    return [
        # the smallest job: one workgroup's worth of state, 720 gates, 1024 shots
        {"name": "shots_12", "kind": "shots", "n": 12, "layers": 40, "shots": 1024},
        # a circuit of QASMBench's middle sizes, handed over as text
        {"name": "job_16", "kind": "job", "n": 16, "layers": 24, "shots": 1024},
        # a host program that keeps its own state: both copies and a short circuit
        {"name": "state_21", "kind": "state", "n": 21, "layers": 10},
        # the headline circuit: 890 gates on a state of 16 GiB
        {"name": "xeb_30", "kind": "xeb", "n": 30, "layers": 20, "shots": 4096},
        # the largest state (32 GiB): phases and swaps
        {"name": "qft_31", "kind": "qft", "n": 31, "shots": 4096, "compiled": False},
        # the same work at an ordinary size, compiled for repeated runs
        {"name": "qft_27_compiled", "kind": "qft", "n": 27, "shots": 4096, "compiled": True},
        # a QIR program with 16 mid-circuit measurements
        {"name": "qir_27", "kind": "qir", "n": 27, "gates": 800, "measures": 16},
        # a density matrix of 13 qubits, the most that the reference's engine takes
        {"name": "dm_13", "kind": "dm", "n": 13, "gates": 400, "measures": 4},
        # the energy of an Ising model on a kept state, 55 terms
        {"name": "energy_28", "kind": "energy", "n": 28},
        # a training step of a 320-parameter ansatz
        {"name": "train_20", "kind": "train", "n": 20, "layers": 8},
        # the gradient of a kept circuit on a larger state, odd qubit count
        {"name": "grad_25", "kind": "grad", "n": 25, "layers": 6},
        # many uneven circuits at once
        {"name": "batch_96", "kind": "batch", "count": 96, "nmin": 10, "nmax": 20, "lmin": 2, "lmax": 8},
    ]


def draw(rng):
    kind = rng.choice(["shots", "job", "state", "xeb", "qft", "qir", "dm", "energy", "train", "grad", "batch"])
    u = rng.randint

    def log(lo, hi):   # an integer spread over the logarithm of the range
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "shots":
        return {"kind": kind, "n": u(3, 20), "layers": u(5, 60), "shots": log(16, 8192)}
    if kind == "job":
        return {"kind": kind, "n": u(4, 20), "layers": u(4, 40), "shots": log(16, 8192)}
    if kind == "state":
        return {"kind": kind, "n": u(14, 23), "layers": u(2, 20)}
    if kind == "xeb":
        return {"kind": kind, "n": u(20, 29), "layers": u(6, 24), "shots": log(256, 16384)}
    if kind == "qft":
        return {"kind": kind, "n": u(18, 30), "shots": log(256, 16384), "compiled": rng.random() < 0.25}
    if kind == "qir":
        return {"kind": kind, "n": u(14, 28), "gates": u(100, 800), "measures": u(1, 16)}
    if kind == "dm":
        return {"kind": kind, "n": u(6, 13), "gates": u(60, 400), "measures": u(1, 4)}
    if kind == "energy":
        return {"kind": kind, "n": u(16, 28)}
    if kind == "train":
        return {"kind": kind, "n": u(8, 22), "layers": u(2, 10)}
    if kind == "grad":
        return {"kind": kind, "n": u(12, 25), "layers": u(2, 8)}
    lo = u(6, 12)
    return {"kind": kind, "count": log(8, 128), "nmin": lo, "nmax": lo + u(2, 8), "lmin": 2, "lmax": u(3, 10)}


# ------------------------------------------------------------------ circuits
#
# Gates as (name, qubits, angles...), the form from which both the engine's
# records and the plain torch simulation are made.


def _layers(n, layers, rng):
    gates = []
    for _ in range(layers):
        kinds, ang = rng.integers(0, 4, size=n), rng.random(n) * 2 * np.pi
        for q in range(n):
            k = ("H", "RX", "RY", "RZ")[kinds[q]]
            gates.append((k, (q,)) if k == "H" else (k, (q,), float(ang[q])))
        perm = rng.permutation(n)
        for i in range(0, n - 1, 2):
            gates.append(("CX", (int(perm[i]), int(perm[i + 1]))))
    return gates


def _brickwall(n, layers, rng):
    gates = []
    for l in range(layers):
        ang = rng.random((n, 3)) * 2 * np.pi
        for q in range(n):
            gates.append(("U3", (q,), *(float(a) for a in ang[q])))
        for i in range(l % 2, n - 1, 2):
            gates.append(("CZ", (i, i + 1)))
    return gates


def _qft(n):
    gates = []
    for i in range(n):
        gates.append(("H", (i,)))
        for k in range(1, n - i):
            gates.append(("CU1", (i + k, i), math.pi / 2 ** k))
    return gates + [("SWAP", (i, n - 1 - i)) for i in range(n // 2)]


def _ansatz(n, layers, rng):
    """Layers of RY and RZ on every qubit, then a CX ladder; every angle is a parameter."""
    gates = []
    for _ in range(layers):
        ang = rng.random(2 * n) * 2 * np.pi - np.pi
        gates += [("RY", (q,), float(ang[q])) for q in range(n)]
        gates += [("RZ", (q,), float(ang[n + q])) for q in range(n)]
        gates += [("CX", (q, q + 1)) for q in range(n - 1)]
    return gates


def _ising(n, rng):
    J, h = rng.standard_normal(n - 1), rng.standard_normal(n)
    return ([(float(J[i]), 0, (1 << i) | (1 << (i + 1))) for i in range(n - 1)]
            + [(float(h[i]), 1 << i, 0) for i in range(n)])


def _job_gates(n, layers, rng):
    """What a QASM file holds: one-qubit rotations, U3, CX, CZ, controlled phases and Toffolis."""
    gates = []
    for _ in range(layers):
        for q in range(n):
            k = ("H", "RX", "RY", "RZ", "U3")[int(rng.integers(5))]
            ang = [float(a) for a in rng.random(3) * 2 * np.pi]
            gates.append((k, (q,), *ang[:{"H": 0, "U3": 3}.get(k, 1)]))
        perm = [int(q) for q in rng.permutation(n)]
        for i in range(0, n - 2, 3):
            k = ("CX", "CZ", "CU1", "CCX")[int(rng.integers(4))]
            qs = tuple(perm[i:i + 3]) if k == "CCX" else tuple(perm[i:i + 2])
            gates.append((k, qs, float(rng.random() * 2 * np.pi)) if k == "CU1" else (k, qs))
    return gates


def _qasm_text(n, gates):
    lines = ["OPENQASM 2.0;", 'include "qelib1.inc";', "qreg q[%d];" % n, "creg c[%d];" % n]
    for name, qs, *ang in gates:
        args = "(%s)" % ",".join(repr(a) for a in ang) if ang else ""
        lines.append("%s%s %s;" % (name.lower(), args, ",".join("q[%d]" % q for q in qs)))
    lines += ["measure q[%d] -> c[%d];" % (q, q) for q in range(n)]
    return "\n".join(lines) + "\n"


_FIELD = {"RX": ("theta",), "RY": ("theta",), "RZ": ("phi",), "U3": ("theta", "phi", "lambda"), "CU1": ("lambda",)}


def _records(gates):
    import svmi
    arr = np.zeros(len(gates), dtype=svmi.GATE_DTYPE)
    for r, (name, qs, *ang) in zip(arr, gates):
        r["op"] = svmi.OP[name]
        r["qb"][:len(qs)] = qs
        for f, a in zip(_FIELD.get(name, ()), ang):
            r[f] = a
    return arr


def _slots(gates):
    """Parameter of each gate's (theta, phi, lambda): one for every rotation, in order."""
    s, p = np.full((len(gates), 3), -1, dtype=np.int32), 0
    for i, g in enumerate(gates):
        if g[0] in ("RY", "RZ"):
            s[i, 0 if g[0] == "RY" else 1] = p
            p += 1
    return s, p


_QIR1 = ("X", "Y", "Z", "H", "S", "T", "RI", "RX", "RY", "RZ", "EI", "EX", "EY", "EZ", "AdjointS", "AdjointT")


def _qir_program(n, count, measures, rng):
    """(op, qubit, mask, angle) records: 60 % one-qubit gates, 30 % with 1-3 controls, 5 % X or Z
    controlled by all other qubits, 5 % Swap, and measurements in the Z, X and Y bases in turn."""
    rows, m, every = [], 0, max(1, count // measures)
    for i in range(count):
        q = int(rng.integers(n))
        if (i + 1) % every == 0 and m < measures:
            rows.append(("Measure", q, m % 3, int(rng.integers(0, _RAND_MAX)) / _RAND_MAX))
            m += 1
            continue
        u, theta = rng.random(), float(rng.uniform(-2 * np.pi, 2 * np.pi))
        others = [c for c in range(n) if c != q]
        if u < 0.60:
            rows.append((_QIR1[int(rng.integers(len(_QIR1)))], q, 0, theta))
        elif u < 0.90:
            mask = sum(1 << int(c) for c in rng.choice(others, size=int(rng.integers(1, 4)), replace=False))
            name = _QIR1[int(rng.integers(len(_QIR1)))]
            rows.append(("Controlled" + name, q, mask, theta))
        elif u < 0.95:
            rows.append((("ControlledX", "ControlledZ")[int(rng.integers(2))], q, ((1 << n) - 1) & ~(1 << q), 0.0))
        else:
            rows.append(("Swap", q, int(rng.choice(others)), 0.0))
    return rows


def _uniforms(shots, rng):
    """Draws rand() / RAND_MAX, as the reference's measure() makes them."""
    return rng.integers(0, _RAND_MAX, size=shots).astype(np.float64) / _RAND_MAX


def _host_state(n, rng):
    re, im = rng.standard_normal(1 << n), rng.standard_normal(1 << n)
    s = math.sqrt(float(re @ re + im @ im))
    return re / s, im / s


def _inputs(case, seed):
    """The case's inputs as plain values: the same for the engine and for exact()."""
    rng = np.random.default_rng([seed, 77])
    k, n = case["kind"], case.get("n")
    if k == "shots":
        return {"gates": _layers(n, case["layers"], rng), "u": _uniforms(case["shots"], rng)}
    if k == "job":
        return {"gates": _job_gates(n, case["layers"], rng), "u": _uniforms(case["shots"], rng)}
    if k == "state":
        return {"gates": _layers(n, case["layers"], rng), "state": _host_state(n, rng)}
    if k in ("xeb", "qft"):
        gates = _brickwall(n, case["layers"], rng) if k == "xeb" else _qft(n)
        return {"gates": gates, "u": _uniforms(case["shots"], rng),
                "idx": rng.integers(0, 1 << n, size=_AMPS).astype(np.uint64), "seed": 1 + int(rng.integers(1 << 40))}
    if k in ("qir", "dm"):
        bits = n if k == "qir" else 2 * n
        return {"rows": _qir_program(n, case["gates"], case["measures"], rng),
                "idx": rng.integers(0, 1 << bits, size=min(_AMPS, 1 << bits)).astype(np.uint64)}
    if k == "energy":
        return {"terms": _ising(n, rng), "seed": 1 + int(rng.integers(1 << 40))}
    if k in ("train", "grad"):
        return {"gates": _ansatz(n, case["layers"], rng), "terms": _ising(n, rng)}
    # the sizes are the case's, the angles and couplings the seed's
    sizes = np.random.default_rng([case[f] for f in ("count", "nmin", "nmax", "lmin", "lmax")])
    items = []
    for _ in range(case["count"]):
        m, l = int(sizes.integers(case["nmin"], case["nmax"] + 1)), int(sizes.integers(case["lmin"], case["lmax"] + 1))
        items.append({"n": m, "gates": _ansatz(m, l, rng), "terms": _ising(m, rng)})
    return {"items": items}


# ------------------------------------------------------- prepare, run, work


def prepare(case, seed):
    import svmi
    x, k = _inputs(case, seed), case["kind"]
    s = {"kind": k, "x": x}
    if k == "batch":
        s["items"] = []
        for it in x["items"]:
            slots, p = _slots(it["gates"])
            s["items"].append({"n": it["n"], "gates": _records(it["gates"]), "param_slots": slots, "n_params": p,
                               "terms": svmi.as_terms(it["terms"])})
        return s
    if k == "train":
        from svmi.autograd import ExpvalCircuit
        slots, p = _slots(x["gates"])
        s["circuit"] = ExpvalCircuit(case["n"], _records(x["gates"]), slots, p, svmi.as_terms(x["terms"]))
        s["params"] = torch.tensor([g[2] for g in x["gates"] if len(g) > 2], dtype=torch.float64, requires_grad=True)
        return s
    e = s["engine"] = svmi.Engine(2 * case["n"] if k == "dm" else case["n"])
    if k == "job":
        s["text"] = _qasm_text(case["n"], x["gates"])
    elif k in ("qir", "dm"):
        s["n"], s["rows"] = case["n"], svmi.as_qir_gates(x["rows"])
    elif k == "energy":
        e.set_random_state(x["seed"])
        s["terms"] = svmi.as_terms(x["terms"])
    else:
        if case.get("compiled"):
            e.set_option(svmi.OPT_SPECIALIZE, 1)
        e.upload(_records(x["gates"]))
        if k == "qft":
            e.set_random_state(x["seed"])
        if k == "grad":
            s["slots"], s["n_params"] = _slots(x["gates"])
            s["terms"] = svmi.as_terms(x["terms"])
    return s


def run(s):
    k, x, e = s["kind"], s["x"], s.get("engine")
    if k == "batch":
        import svmi
        ev, grads = svmi.batch_adjoint(s["items"])
        return {"energies": ev, "grads": np.concatenate(grads)}
    if k == "train":
        p = s["params"]
        p.grad = None
        energy = s["circuit"](p)
        energy.backward()
        with torch.no_grad():
            p.sub_(p.grad, alpha=0.02)
        return {"energy": energy.detach(), "grad": p.grad, "params": p.detach().clone()}
    if k == "energy":
        return {"energy": e.expval(s["terms"])}
    if k == "grad":
        e.reset_state()
        energy, grad = e.adjoint(s["terms"], s["slots"], s["n_params"])
        return {"energy": energy, "grad": grad}
    if k in ("qir", "dm"):
        e.reset_state()
        r = e.qir_run(s["n"], s["rows"]) if k == "qir" else e.dm_qir_run(s["n"], s["rows"])
        re, im = e.get_amplitudes(x["idx"])
        return {"probs": r[0], "outcomes": r[1], "re": re, "im": im}
    if k == "state":
        e.set_state(*x["state"])
        e.run()
        re, im = e.get_state()
        return {"re": re, "im": im}
    if k == "job":
        from svmi import qasm
        _, gates, _ = qasm.parse(s["text"])
        e.upload(gates)
    if k != "qft":
        e.reset_state()
    e.run()
    shots, total = e.measure(x["u"])
    re, im = e.get_state() if k in ("shots", "job") else e.get_amplitudes(x["idx"])
    return {"shots": shots.astype(np.int64), "total": total, "re": re, "im": im}


def work(case):
    """The state read once and written once where a circuit runs on it (twice for a gradient: the
    state and its adjoint), and read once for samples or an energy; the host's copies where there
    are any.  Operations: 14 for each amplitude and one-qubit gate (a 2x2 of complex numbers), 6 for
    each amplitude that a phase turns."""
    k = case["kind"]
    if k == "batch":
        n = (case["nmin"] + case["nmax"]) / 2
        amp = case["count"] * 2 ** (case["nmax"] + 1) / (case["nmax"] - case["nmin"] + 1)   # mean of 2^n
        return {"bytes": 96 * amp, "flops": amp * 3 * 2 * n * 14 * (case["lmin"] + case["lmax"]) / 2}
    n = case["n"]
    amp = 2 ** (2 * n if k == "dm" else n)
    if k == "energy":
        return {"bytes": 16 * amp, "flops": amp * (n * 4 + 6)}
    if k in ("train", "grad"):
        return {"bytes": 96 * amp, "flops": amp * 3 * 2 * n * 14 * case["layers"]}
    if k == "state":
        return {"bytes": 64 * amp, "flops": amp * n * 14 * case["layers"]}
    if k in ("qir", "dm"):
        return {"bytes": 32 * amp, "flops": amp * 10 * case["gates"] * (2 if k == "dm" else 1)}
    gates = {"qft": n * 14 + n * (n - 1) * 3 / 4}.get(k) or n * 14 * case["layers"]
    return {"bytes": 48 * amp, "flops": amp * gates}


# ------------------------------------------- the same in plain torch, 64 bits


def _sub(psi, n, fixed):
    """View of psi's amplitudes whose qubits have the given bits ({qubit: bit})."""
    off, size, stride, q = 0, [], [], 0
    while q < n:
        if q in fixed:
            off += fixed[q] << q
            q += 1
            continue
        q0 = q
        while q < n and q not in fixed:
            q += 1
        size.insert(0, 1 << (q - q0))
        stride.insert(0, 1 << q0)
    return torch.as_strided(psi, size or [1], stride or [1], off)


def _mat(psi, n, q, m, ctrl=()):
    """2x2 matrix m on qubit q where all qubits of ctrl are 1."""
    c = {t: 1 for t in ctrl}
    b = _sub(psi, n, {**c, q: 1})
    if m[0][1] == 0 and m[1][0] == 0:
        if m[0][0] != 1:
            _sub(psi, n, {**c, q: 0}).mul_(m[0][0])
        if m[1][1] != 1:
            b.mul_(m[1][1])
        return
    a = _sub(psi, n, {**c, q: 0})
    t = a * m[0][0]
    t.add_(b, alpha=m[0][1])
    b.mul_(m[1][1]).add_(a, alpha=m[1][0])
    a.copy_(t)


def _e(t):
    return complex(math.cos(t), math.sin(t))


def _matrix(name, ang):
    """The 2x2 of a gate; RZ is the reference's, which turns only the |1> amplitude."""
    r = math.sqrt(0.5)
    if name == "H":
        return [[r, r], [r, -r]]
    if name in ("X", "CX", "CCX"):
        return [[0, 1], [1, 0]]
    if name == "CZ":
        return [[1, 0], [0, -1]]
    if name in ("RZ", "CU1"):
        return [[1, 0], [0, _e(ang[0])]]
    c, s = math.cos(ang[0] / 2), math.sin(ang[0] / 2)
    if name == "RX":
        return [[c, -1j * s], [-1j * s, c]]
    if name == "RY":
        return [[c, -s], [s, c]]
    return [[c, -_e(ang[2]) * s], [_e(ang[1]) * s, _e(ang[1] + ang[2]) * c]]   # U3


def _gate(psi, n, g):
    name, qs, *ang = g
    if name == "SWAP":
        a, b = _sub(psi, n, {qs[0]: 0, qs[1]: 1}), _sub(psi, n, {qs[0]: 1, qs[1]: 0})
        t = a.clone()
        a.copy_(b)
        b.copy_(t)
    else:
        _mat(psi, n, qs[-1], _matrix(name, ang), qs[:-1])


def _zero(n, dev):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=dev)
    psi[0] = 1
    return psi


def _c(m, dev):
    return torch.tensor(m, dtype=torch.complex128, device=dev)


def _run_brickwall(psi, n, gates, dev):
    """The U3s of a layer five qubits at a time as one 32x32 product: the rest is sign flips."""
    layer = []
    for g in gates + [None]:
        if g is not None and g[0] == "U3":
            layer.append(g)
            continue
        for i in range(0, len(layer), 5):
            K = torch.ones(1, 1, dtype=torch.complex128, device=dev)
            for h in layer[i:i + 5]:
                K = torch.kron(_c(_matrix("U3", h[2:]), dev), K)
            # the lowest qubits of the index, which then become its highest
            psi = (psi.view(-1, K.shape[0]) @ K.T.contiguous()).t().contiguous().view(-1)
        layer = []
        if g is not None:
            _gate(psi, n, g)
    return psi


def _run_qft(psi, n, dev):
    for i in range(n):
        _mat(psi, n, i, _matrix("H", ()))
        if i + 1 < n:   # the controlled phases of qubit i as one factor over the qubits above it
            w = torch.ones(1, dtype=torch.complex128, device=dev)
            for k in range(1, n - i):
                w = torch.cat([w, w * _e(math.pi / 2 ** k)])
            psi.view(-1, 2, 1 << i)[:, 1].mul_(w[:, None])
    for i in range(n // 2):
        _gate(psi, n, ("SWAP", (i, n - 1 - i)))
    return psi


def _i64(v):
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    """splitmix64 on int64 tensors."""
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _i64(0x94D049BB133111EB)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _seeded_state(n, seed, dev):
    """The documented seeded random state: Box-Muller of two splitmix64 uniforms per amplitude."""
    psi = torch.empty(1 << n, dtype=torch.complex128, device=dev)
    norm, step = 0.0, 1 << min(n, 24)
    for x0 in range(0, 1 << n, step):
        x = torch.arange(x0, x0 + step, dtype=torch.int64, device=dev) * 2 + seed
        u = [(((_mix(x + k) >> 11) & ((1 << 53) - 1)) + 1).double() * 2.0 ** -53 for k in (1, 2)]
        r, t = torch.sqrt(-2 * torch.log(u[0])), 2 * math.pi * u[1]
        psi[x0:x0 + step] = torch.complex(r * torch.cos(t), r * torch.sin(t))
        norm += float((r * r).sum())
    return psi.mul_(1 / math.sqrt(norm))


def _h_psi(psi, n, terms):
    """H psi for sums of Z strings and single X."""
    d = torch.zeros(1 << n, dtype=torch.float64, device=psi.device)
    lam = torch.zeros_like(psi)
    for c, xm, zm in terms:
        if xm:
            q = xm.bit_length() - 1
            for b in (0, 1):
                _sub(lam, n, {q: b}).add_(_sub(psi, n, {q: 1 - b}), alpha=c)
        else:
            i, j = (q for q in range(n) if (zm >> q) & 1)
            for b in range(4):
                _sub(d, n, {i: b & 1, j: b >> 1}).add_(c if b in (0, 3) else -c)
    return lam.addcmul_(psi, d.to(psi.dtype))


def _gradient(n, gates, terms, dev):
    psi = _zero(n, dev)
    for g in gates:
        _gate(psi, n, g)
    lam = _h_psi(psi, n, terms)
    energy = float(torch.vdot(psi, lam).real)
    grad = []
    for g in reversed(gates):
        name, (*ctrl, q), *ang = g
        m = _matrix(name, ang)
        inv = [[complex(m[j][i]).conjugate() for j in (0, 1)] for i in (0, 1)]
        _mat(psi, n, q, inv, ctrl)
        if ang:
            p0, p1, l0, l1 = (_sub(v, n, {q: b}).reshape(-1) for v in (psi, lam) for b in (0, 1))
            if name == "RY":   # dU = [[-s, -c], [c, -s]] / 2
                c, s = math.cos(ang[0] / 2), math.sin(ang[0] / 2)
                v = -s * (torch.vdot(l0, p0) + torch.vdot(l1, p1)) + c * (torch.vdot(l1, p0) - torch.vdot(l0, p1))
                grad.append(float(v.real))
            else:              # dU = diag(0, i exp(i phi))
                grad.append(2 * float((1j * _e(ang[0]) * torch.vdot(l1, p1)).real))
        _mat(lam, n, q, inv, ctrl)
    return energy, np.array(grad[::-1])


def _qir_matrix(name, t):
    r = math.sqrt(0.5)
    c, s = math.cos(t / 2), math.sin(t / 2)
    C, S = math.cos(t), math.sin(t)
    return {"X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]], "H": [[r, r], [r, -r]],
            "S": [[1, 0], [0, 1j]], "T": [[1, 0], [0, complex(r, r)]], "AdjointS": [[1, 0], [0, -1j]],
            "AdjointT": [[1, 0], [0, complex(r, -r)]], "RI": [[_e(-t / 2), 0], [0, _e(-t / 2)]],
            "RX": [[c, -1j * s], [-1j * s, c]], "RY": [[c, -s], [s, c]], "RZ": [[_e(-t / 2), 0], [0, _e(t / 2)]],
            "EI": [[_e(t), 0], [0, _e(t)]], "EX": [[C, 1j * S], [1j * S, C]], "EY": [[C, S], [-S, C]],
            "EZ": [[_e(t), 0], [0, _e(-t)]]}[name]


def _run_qir(n, rows, dm, dev):
    """The records on a state of n qubits, or as U and conj(U) on the rows and columns of a density
    matrix (index row | column << n), whose Swap and collapse touch the rows only."""
    bits = 2 * n if dm else n
    psi, probs = _zero(bits, dev), []

    def both(name, q, t, ctrl=()):
        m = _qir_matrix(name, t)
        _mat(psi, bits, q, m, ctrl)
        if dm:
            _mat(psi, bits, q + n, [[complex(v).conjugate() for v in r] for r in m], [c + n for c in ctrl])

    for name, q, mask, t in rows:
        if name == "Swap":
            _gate(psi, bits, ("SWAP", (q, mask)))
        elif name == "Measure":
            for b in (["H"], ["AdjointS", "H"])[mask - 1] if mask else []:
                both(b, q, 0.0)
            if dm:
                d = psi[:: (1 << n) + 1].real.abs()
                p = float(_sub(d.contiguous(), n, {q: 1}).sum())
            else:
                p = float(_sub(psi, n, {q: 1}).abs().square().sum())
            probs.append(p)
            one = 1 if t < p else 0
            w = p if one else 1 - p
            _sub(psi, bits, {q: 1 - one}).zero_()
            _sub(psi, bits, {q: one}).mul_(1 / w if dm else 1 / math.sqrt(w))
            for b in (["H"], ["H", "S"])[mask - 1] if mask else []:
                both(b, q, 0.0)
        elif name.startswith("Controlled"):
            both(name[10:], q, t, [c for c in range(n) if (mask >> c) & 1])
        else:
            both(name, q, t)
    return psi, probs


def exact(case, seed):
    x, k, n = _inputs(case, seed), case["kind"], case.get("n")
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if k == "batch":
        if sum(len(it["gates"]) for it in x["items"]) > 40000:
            return None
        got = [_gradient(it["n"], it["gates"], it["terms"], dev) for it in x["items"]]
        return {"energies": np.array([e for e, _ in got]), "grads": np.concatenate([g for _, g in got])}
    if k in ("train", "grad"):
        energy, grad = _gradient(n, x["gates"], x["terms"], dev)
        if k == "grad":
            return {"energy": energy, "grad": grad}
        p = np.array([g[2] for g in x["gates"] if len(g) > 2])
        return {"energy": torch.tensor(energy, dtype=torch.float64), "grad": torch.from_numpy(grad),
                "params": torch.from_numpy(p - 0.02 * grad)}
    if k == "energy":
        psi = _seeded_state(n, x["seed"], dev)
        return {"energy": float(torch.vdot(psi, _h_psi(psi, n, x["terms"])).real)}
    if k in ("qir", "dm"):
        psi, probs = _run_qir(n, x["rows"], k == "dm", dev)
        v = psi[torch.from_numpy(x["idx"].astype(np.int64)).to(dev)].cpu().numpy()
        return {"probs": np.array(probs), "outcomes": None, "re": v.real.copy(), "im": v.imag.copy()}
    if k == "xeb":
        psi = _run_brickwall(_zero(n, dev), n, x["gates"], dev)
    elif k == "qft":
        psi = _run_qft(_seeded_state(n, x["seed"], dev), n, dev)
    else:
        psi = _zero(n, dev)
        if k == "state":
            psi = torch.complex(*(torch.from_numpy(v) for v in x["state"])).to(dev)
        for g in x["gates"]:
            _gate(psi, n, g)
    if k == "state":
        v = psi.cpu().numpy()
        return {"re": v.real.copy(), "im": v.imag.copy()}
    total = float(torch.linalg.vector_norm(psi) ** 2)
    if k in ("xeb", "qft"):
        psi = psi[torch.from_numpy(x["idx"].astype(np.int64)).to(dev)]
    v = psi.cpu().numpy()
    return {"shots": None, "total": total, "re": v.real.copy(), "im": v.imag.copy()}
