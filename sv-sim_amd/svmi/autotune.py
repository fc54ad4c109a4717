"""Autotuner of batched planning.

For each qubit count n it times `svmi.batch_adjoint` (expectation + adjoint
gradient, planning included) on a batch of hardware-efficient-ansatz circuits
of that size -- the gate pattern and observable of the batched workload, layer
counts 2..10 -- and picks, by coordinate descent from the single-circuit
settings, the fusion op cost, then the forward sweep tile, then the backward
sweep tile (below 18 qubits: from there on the engine's own is 12, more than an
item can ask for, and every candidate runs with it).  A candidate replaces the
current choice only when it is more than 3 % faster (median of 3 runs).  The
result is written as the C++ table sv-sim_amd/csrc/svmi_tuning.hpp (rebuild the
library afterwards) and a JSON log of every measurement.  Batches of one size
say little about mixed ones: compare the two tables there before the new one
stays (--out writes it elsewhere).

  python -m svmi.autotune [--nmin 4] [--nmax 22] [--out PATH] [--json PATH]

Needs a GPU; takes a few minutes.
"""
import argparse
import json
import os
import time

import numpy as np

import svmi
from svmi import workloads as W

HERE = os.path.dirname(os.path.abspath(__file__))
DEFAULT_OUT = os.path.join(os.path.dirname(HERE), "csrc", "svmi_tuning.hpp")
MAX_N = 30
LARGE_ADJ = 18   # kBatchLargeAdj (csrc/svmi_internal.hpp)


def default(n):
    """The single-circuit settings."""
    return {"fwd_tile": 13 if n >= 21 else 12, "adj_tile": 11, "op_cost": 2}


def batch_for(n, seed):
    """Ansatz circuits of n qubits, layers 2..10, enough of them for a few ms of work."""
    rng = np.random.default_rng(seed)
    count = int(min(64, max(4, (1 << 24) >> n)))
    items = []
    for _ in range(count):
        layers = int(rng.integers(2, 11))
        gates, slots, p = W.hea(n, layers, rng)
        items.append({"n": n, "gates": gates, "param_slots": slots, "n_params": p, "terms": W.ising_terms(n, rng)})
    return items


def time_batch(items, setting, reps=3):
    if items[0]["n"] >= LARGE_ADJ:
        setting = dict(setting, adj_tile=0)
    run = [dict(it, **setting) for it in items]
    svmi.batch_adjoint(run)
    ts = []
    for _ in range(reps):
        t0 = time.perf_counter()
        svmi.batch_adjoint(run)
        ts.append(time.perf_counter() - t0)
    return float(np.median(ts))


def tune_n(n, log):
    items = batch_for(n, seed=9000 + n)
    best = default(n)
    best_t = time_batch(items, best)
    log.append({"n": n, "setting": dict(best), "ms": best_t * 1e3})
    space = {
        "op_cost": [0, 1, 2, 4, 8],
        "fwd_tile": sorted({min(k, max(n, 4)) for k in (6, 8, 10, 12, 13)}),
        "adj_tile": sorted({min(k, max(n, 4)) for k in (6, 8, 9, 10, 11)}) if n < LARGE_ADJ else [],
    }
    for key in ("op_cost", "fwd_tile", "adj_tile"):
        for v in space[key]:
            if v == best[key]:
                continue
            cand = dict(best, **{key: v})
            t = time_batch(items, cand)
            log.append({"n": n, "setting": cand, "ms": t * 1e3})
            if t < 0.97 * best_t:
                best, best_t = cand, t
    print(f"n={n}: {best} {best_t * 1e3:.2f} ms ({len(items)} circuits)", flush=True)
    return best, best_t


def write_header(path, table, source):
    rows = []
    for n in range(4, MAX_N + 1):
        e = table.get(n, default(n))
        rows.append(f"{{{n}, {e['fwd_tile']}, {e['adj_tile']}, {e['op_cost']}}}")
    body = ",\n    ".join(", ".join(rows[i:i + 6]) for i in range(0, len(rows), 6))
    text = f'''// svmi_tuning.hpp -- planning of batched circuits per qubit count.
// Generated by svmi/autotune.py: {source}.
// Sizes outside the tuned range keep the single-circuit settings.  From
// kBatchLargeAdj qubits on adj_tile is not read.
#pragma once

#include <stdint.h>

namespace svmi {{

struct BatchTuning {{
    uint8_t n;          // qubits
    uint8_t fwd_tile;   // forward sweep tile qubits
    uint8_t adj_tile;   // backward sweep tile qubits
    uint8_t op_cost;    // fusion op cost
}};

constexpr const char* kBatchTuningSource = "{source}";
constexpr BatchTuning kBatchTuning[] = {{
    {body},
}};

// Entry for an n-qubit circuit (the nearest size in the table).
inline const BatchTuning& batch_tuning(int n)
{{
    constexpr int count = int(sizeof(kBatchTuning) / sizeof(kBatchTuning[0]));
    int best = 0;
    for (int i = 1; i < count; i++) {{
        const int d = n - int(kBatchTuning[i].n), db = n - int(kBatchTuning[best].n);
        if ((d < 0 ? -d : d) < (db < 0 ? -db : db)) best = i;
    }}
    return kBatchTuning[best];
}}

}}  // namespace svmi
'''
    with open(path, "w") as f:
        f.write(text)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--nmin", type=int, default=4)
    ap.add_argument("--nmax", type=int, default=22)
    ap.add_argument("--out", default=DEFAULT_OUT)
    ap.add_argument("--json", default=None)
    a = ap.parse_args()
    import torch
    if not torch.cuda.is_available():
        raise SystemExit("autotune needs a GPU")
    dev = torch.cuda.get_device_properties(0)
    arch = getattr(dev, "gcnArchName", "").split(":")[0]
    table, log = {}, []
    for n in range(a.nmin, a.nmax + 1):
        table[n], _ = tune_n(n, log)
    source = f"{dev.name} ({arch}), n = {a.nmin}..{a.nmax}, {time.strftime('%Y-%m-%d')}"
    write_header(a.out, table, source)
    if a.json:
        with open(a.json, "w") as f:
            json.dump({"source": source, "table": table, "runs": log}, f, indent=1)
    print(f"wrote {a.out}", flush=True)


if __name__ == "__main__":
    main()
