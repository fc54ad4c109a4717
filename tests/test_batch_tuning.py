"""The batch tuner measures what the table's users get: an item that asks for
the table's own tiles and op cost plans as one that asks for nothing (the same
sums in the same order: bit-equal results), and what an item could not ask for
is refused as before."""
import os
import re

import numpy as np
import pytest

import svmi
from svmi import autotune
from svmi import workloads as W

HEADER = os.path.join(os.path.dirname(__file__), "..", "sv-sim_amd", "csrc", "svmi_tuning.hpp")


def _rows():
    return {int(n): {"fwd_tile": int(f), "adj_tile": int(a), "op_cost": int(c)}
            for n, f, a, c in re.findall(r"\{(\d+), (\d+), (\d+), (\d+)\}", open(HEADER).read())}


def _item(n, layers, seed):
    rng = np.random.default_rng(seed)
    gates, slots, p = W.hea(n, layers, rng)
    return {"n": n, "gates": gates, "param_slots": slots, "n_params": p, "terms": W.ising_terms(n, rng)}


@pytest.mark.parametrize("n,layers", [(4, 3), (8, 3), (9, 2), (12, 2), (13, 2), (14, 2), (18, 1)])
def test_asking_for_the_table_is_the_default(n, layers):
    it, row = _item(n, layers, n), dict(_rows()[n])
    if n >= autotune.LARGE_ADJ:
        row["adj_tile"] = 0   # the engine's own, as the tuner measures it
    e0, g0 = svmi.emulate_batch([it])
    e1, g1 = svmi.emulate_batch([dict(it, **row)])
    assert e0[0] == e1[0] and np.array_equal(g0[0], g1[0])


def test_tuner_settings_match_the_engine():
    src = open(os.path.join(os.path.dirname(HEADER), "svmi_internal.hpp")).read()
    assert int(re.search(r"kBatchLargeAdj = (\d+)", src).group(1)) == autotune.LARGE_ADJ


@pytest.mark.parametrize("kw", [{"fwd_tile": 5}, {"fwd_tile": 4}, {"adj_tile": 5}])
def test_tiles_too_small_for_an_op_stay_refused(kw):
    c = W.Circuit()
    c.add("SWAP", [5, 6])   # beside the 4 low qubits it needs 6
    it = {"n": 7, "gates": c.array(), "param_slots": np.full((1, 3), -1, dtype=np.int32), "n_params": 0,
          "terms": [(1.0, 0, 1)]}
    with pytest.raises(svmi.SvmiError, match="does not fit a tile"):
        svmi.emulate_batch([dict(it, **kw)])
