"""GPU: an upload's host copy of the program's tables does not stay with the
handle: what glibc has given out is back near the start once the circuit is
cleared."""
import ctypes

import numpy as np
import pytest

import svmi
from svmi import workloads as W

pytestmark = pytest.mark.gpu


class _Mallinfo2(ctypes.Structure):
    _fields_ = [(f, ctypes.c_size_t) for f in ("arena", "ordblks", "smblks", "hblks", "hblkhd", "usmblks", "fsmblks",
                                               "uordblks", "fordblks", "keepcost")]


def _in_use():
    f = ctypes.CDLL(None).mallinfo2
    f.restype = _Mallinfo2
    m = f()
    return m.uordblks + m.hblkhd


def test_upload_keeps_no_copy_of_a_large_program():
    n = 22
    large = W.u3_brickwall(n, 600)
    with svmi.Engine(n) as e:   # what the runtime keeps from a first large copy is not the engine's
        e.upload(large)
    with svmi.Engine(n) as e:
        base = _in_use()
        e.upload(large)
        held = _in_use() - base
        e.clear_circuit()
        left = _in_use() - base
    assert held > 6 << 20          # the program itself, while the circuit is there
    assert left < 2 << 20          # 1 MiB may be kept for the next upload, and the gate list's capacity
