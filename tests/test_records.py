"""Angles of recorded gates that are not finite: refused where the gate's
matrix is, planned where it holds NaN."""

import ctypes

import numpy as np
import pytest

from qibojit_amd import _native
from qibojit_amd._qibo import gates
from qibojit_amd.backends.matrices import KernelMatrices
from qibojit_amd.fusion import target_block
from qibojit_amd.records import GATE_CODES, Records

INF, NAN = float("inf"), float("nan")
NAMES = sorted(name for name, (_, count) in GATE_CODES.items() if count)


def _plan(gate, encode):
    """Plans the one-gate list (no state, no launch)."""
    records = Records()
    records.add(gate, encode)
    _native.call("qj_run_gates", None, 1, None, _native.QJ_COMPLEX128, 6, 0, 5, 1, records.words.buffer_info()[0],
                 len(records.words), records.params.buffer_info()[0], len(records.params), ctypes.byref(ctypes.c_int32()),
                 None)


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("value", [INF, -INF, NAN, np.float64(INF), 1e308, 10**400])
@pytest.mark.parametrize("name", NAMES)
def test_refused_as_the_matrix_is(name, value):
    encode = KernelMatrices("complex128").encode
    count = GATE_CODES[name][1]
    for place in range(count):
        angles = [0.3] * count
        angles[place] = value
        gate = getattr(gates, name)(*range(2 if name.startswith("C") else 1), *angles)
        try:
            target_block(encode, gate)
        except (ValueError, OverflowError) as error:
            with pytest.raises(type(error)):
                _plan(gate, encode)
        else:
            _plan(gate, encode)
