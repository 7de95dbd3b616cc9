"""Tile passes whose plan travels with the launch, and ones whose plan does
not fit the kernel's arguments (about 32 single-qubit matrices)."""

import numpy as np
import pytest

from qibojit_amd._qibo import Circuit, gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nqubits", [5, 12, 14])
@pytest.mark.parametrize("count", [1, 8, 26, 28, 30, 32, 34, 36, 40, 90])
def test_gate_counts_around_the_argument_size(hip_backend, nqubits, count, dtype):
    hip_backend.set_dtype(dtype)
    rng = np.random.default_rng(count)
    circuit = Circuit(nqubits)
    state = None
    for i in range(count):
        q = int(rng.integers(nqubits))
        p = (q + 1) % nqubits
        angles = [float(a) for a in rng.uniform(-3, 3, 3)]
        gate = [gates.U3(q, *angles), gates.CU3(q, p, *angles), gates.CU1(q, p, angles[0])][i % 3]
        circuit.add(gate)
    got = hip_backend.to_numpy(hip_backend.execute_circuit(circuit).state())
    state = hip_backend.zero_state(nqubits)
    for gate in circuit.queue:
        state = hip_backend.apply_gate(gate, state, nqubits)
    tol = 1e-12 if dtype == "complex128" else 1e-5
    np.testing.assert_allclose(got, hip_backend.to_numpy(state), rtol=0, atol=tol)
