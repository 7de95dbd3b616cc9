"""Gate records of the fused executor (``qj_run_gates``).

A record names a gate by code, targets and controls and appends its
parameters to a float64 list; the library plans and encodes from there.
Gates with scalar double-precision parameters go by name, everything else as
the dense matrix of its target block.
"""

from array import array

import numpy as np

from qibojit_amd.fusion import target_block

MAX_TARGETS = 5  # QJ_TILE_MAX_K
DENSE, DENSE_BITS, SWAP = 0, 1, 2  # QJ_GATE_*

# gate class -> (QJ_GATE_* code of its target block, number of parameters)
GATE_CODES = {}
for _code, _count, _names in (
    (3, 0, "X CNOT TOFFOLI"), (4, 0, "Y CY"), (5, 0, "Z CZ CCZ"), (6, 0, "H CH"), (7, 0, "S"), (8, 0, "SDG"),
    (9, 0, "T"), (10, 0, "TDG"), (11, 0, "SX CSX"), (12, 0, "SXDG CSXDG"), (13, 1, "RX CRX"), (14, 1, "RY CRY"),
    (15, 1, "RZ CRZ"), (16, 1, "U1 CU1"), (17, 2, "U2 CU2"), (18, 3, "U3 CU3"),
):
    for _name in _names.split():
        GATE_CODES[_name] = (_code, _count)

# parameter types evaluated in double precision (a float32 angle keeps its
# single-precision matrix)
_SCALARS = frozenset((float, int, np.float64))


class Records:
    """Records of a run of gates, in order."""

    def __init__(self):
        self.words = array("i")
        self.params = array("d")
        self.count = 0

    def add_dense(self, code, targets, controls, matrix):
        self.words.extend((code, len(targets), len(controls), *targets, *controls))
        self.params.frombytes(np.ascontiguousarray(matrix, dtype=np.complex128).tobytes())
        self.count += 1

    def add(self, gate, custom_matrix_of):
        """Append a unitary gate; False if it is too wide for a tile."""
        name = type(gate).__name__
        targets, controls = gate.target_qubits, gate.control_qubits
        entry = GATE_CODES.get(name)
        if entry is not None:
            code, count = entry
            params = gate.parameters if count else ()
            if len(params) == count and _SCALARS.issuperset(map(type, params)):
                if controls:
                    self.words.extend((code, 1, len(controls), targets[0], *controls))
                else:
                    self.words.extend((code, 1, 0, targets[0]))
                if count:
                    self.params.extend(params)
                self.count += 1
                return True
        elif name == "SWAP" and not controls:
            self.words.extend((SWAP, 2, 0, *targets))
            self.count += 1
            return True
        if len(targets) > MAX_TARGETS:
            return False
        self.add_dense(DENSE, targets, controls, target_block(custom_matrix_of, gate))
        return True

    def clear(self):
        del self.words[:]
        del self.params[:]
        self.count = 0
