"""Passes planned for a QFT: one per tile of high bits and one for the swaps
(in place), or none for the swaps (from another buffer)."""

import ctypes

import numpy as np
import pytest

from qibojit_amd import _native
from qibojit_amd._qibo import gates
from qibojit_amd.records import Records


def _passes(queue, n, dtype, from_source):
    records = Records()
    for gate in queue:
        records.add(gate, None)
    low, high = (6, 7) if dtype == "complex64" else (5, 7)
    code = _native.QJ_COMPLEX64 if dtype == "complex64" else _native.QJ_COMPLEX128
    out = ctypes.c_int32(0)
    _native.call("qj_run_gates", None, int(from_source), None, code, n, 0, low, high, records.words.buffer_info()[0],
                 len(records.words), records.params.buffer_info()[0], len(records.params), ctypes.byref(out), None)
    return out.value


# 26 qubits complex128: the last tile would hold 12 H and 11 ladders, 16.9 KB of
# plan, over the 15 KiB next to a tile; 32 qubits: 11 and 10, which fit
@pytest.mark.parametrize("n,prec,tiles", [(20, "complex64", 2), (30, "complex64", 4), (32, "complex64", 4),
                                           (26, "complex128", 4), (30, "complex128", 4), (32, "complex128", 4)])
def test_qft_passes(n, prec, tiles):
    queue = []
    for q in range(n):
        queue.append(gates.H(q))
        queue += [gates.CU1(p, q, np.pi / 2 ** (p - q)) for p in range(q + 1, n)]
    queue += [gates.SWAP(q, n - 1 - q) for q in range(n // 2)]
    assert _passes(queue, n, prec, False) == tiles + 1
    assert _passes(queue, n, prec, True) == tiles
