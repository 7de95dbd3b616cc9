"""Circuits that end in swaps of many bits, moved to the front and read from
the permuted initial state by the first pass."""

import numpy as np
import pytest

from oracle import gate_matrices as gm
from qibojit_amd._qibo import Circuit, gates

pytestmark = pytest.mark.gpu


def _circuit(n, kind, rng):
    circuit = Circuit(n)
    if kind == "wide":  # a four-qubit matrix on the lowest source bits comes first
        circuit.add(gates.Unitary(gm.haar_unitary(16, rng), 1, n // 2, n // 2 + 1, n - 2))
    if kind == "swaps first":
        for q in range(n // 2):
            circuit.add(gates.SWAP(q, n // 2 + q))
    for q in range(n):
        circuit.add(gates.H(q))
        for p in range(q + 1, n):
            circuit.add(gates.CU1(p, q, float(rng.uniform(-3, 3))))
    if kind != "phase":
        circuit.add(gates.TOFFOLI(0, n - 1, n // 2))
        circuit.add(gates.U3(n - 1, 0.3, 0.7, -0.2))
    for q in range(n // 2):
        circuit.add(gates.SWAP(q, n - 1 - q))
    return circuit


@pytest.mark.parametrize("kernel", ["register", "lds"])
@pytest.mark.parametrize("kind", ["phase", "mixed", "wide", "swaps first"])
@pytest.mark.parametrize("n", [10, 13, 16, 19])
def test_last_swaps_in_the_first_pass(hip_backend, n, kind, kernel, dtype, monkeypatch):
    if kernel == "lds":
        monkeypatch.setenv("QJ_TILE_KERNEL", "lds")
    hip_backend.set_dtype(dtype)
    rng = np.random.default_rng(n)
    circuit = _circuit(n, kind, rng)
    start = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    start /= np.linalg.norm(start)
    tol = 1e-11 if dtype == "complex128" else 2e-5
    for initial in (start, None):
        state = hip_backend.cast(start, copy=True) if initial is not None else hip_backend.zero_state(n)
        initial = None if initial is None else hip_backend.cast(start, copy=True)
        got = hip_backend.to_numpy(hip_backend.execute_circuit(circuit, initial_state=initial).state())
        for gate in circuit.queue:
            state = hip_backend.apply_gate(gate, state, n)
        np.testing.assert_allclose(got, hip_backend.to_numpy(state), rtol=0, atol=tol)
        if initial is not None:  # the source is only read
            np.testing.assert_array_equal(hip_backend.to_numpy(initial), start.astype(dtype))
