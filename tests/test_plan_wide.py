"""Passes planned for five-target gates, which complex128 runs in the LDS
kernel: several a pass where each tile has a CU to itself, with a few other gates
between; passes of their own on larger states and among many other gates."""

import ctypes

import numpy as np
import pytest

from qibojit_amd import _native
from qibojit_amd._qibo import gates
from qibojit_amd.records import Records


def _passes(queue, n):
    records = Records()
    for gate in queue:
        records.add(gate, lambda g: g.parameters[0])
    out = ctypes.c_int32(0)
    _native.call("qj_run_gates", None, 1, None, _native.QJ_COMPLEX128, n, 0, 5, 7, records.words.buffer_info()[0],
                 len(records.words), records.params.buffer_info()[0], len(records.params), ctypes.byref(out), None)
    return out.value


# 16 KiB of matrix each, 128 KiB a pass: seven
@pytest.mark.parametrize("n,others,passes", [(12, 0, 2), (12, 4, 2), (12, 8, 2), (20, 0, 2), (20, 30, 13), (21, 0, 12)])
def test_five_target_passes(n, others, passes):
    u = np.linalg.qr(np.random.default_rng(1).normal(size=(32, 32)))[0]
    queue = []
    for i in range(12):
        queue.append(gates.Unitary(u, *range(n - 5, n)))
        queue += [gates.RX(n - 1 - (i + j) % 5, 0.1) for j in range(others)]
    got = _passes(queue, n)
    assert got == passes if others < 30 else got >= passes
