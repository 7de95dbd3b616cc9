"""Circuits read their starting state in the first pass: results, and the
starting state left as it was, for every kind of first step."""

import numpy as np
import pytest
import torch

from oracle import einsum_ref as er
from oracle import gate_matrices as gm
from qibojit_amd._qibo import Circuit, gates
from tests.conftest import PARITY

pytestmark = pytest.mark.gpu


def _first_steps(n, rng):
    u = gm.haar_unitary(2, rng)
    dense = [(gates.Unitary(u, n - 1), u, (n - 1,)), (gates.H(0), gm.H, (0,))]
    swaps = [(gates.SWAP(i, n - 1 - i), gm.SWAP, (i, n - 1 - i)) for i in range(n // 2)]
    wide = []
    if n >= 6:  # six targets: not a tile op
        w = gm.haar_unitary(64, rng)
        wide = [(gates.Unitary(w, *range(6)), w, tuple(range(6)))]
    return {"dense": dense, "swaps": swaps + dense, "wide": wide + dense, "empty": [],
            "measured": [(gates.M(0), None, ())] + dense, "phase": [(gates.S(0), np.diag([1, 1j]), (0,))]}


@pytest.mark.parametrize("first", ["dense", "swaps", "wide", "empty", "measured", "phase"])
@pytest.mark.parametrize("n", [1, 3, 9, 10, 14])
def test_first_pass_reads_the_start(backend, dtype, n, first, rng):
    backend.set_dtype(dtype)
    steps = _first_steps(n, rng)[first]
    circuit = Circuit(n)
    circuit.add([g for g, _, _ in steps])
    zero = np.zeros(2**n, dtype=complex)
    zero[0] = 1
    for start in (gm.random_state(n, rng, dtype), None):
        want = zero if start is None else start.astype(complex)
        for _, matrix, targets in steps:
            if matrix is not None:
                want = er.apply_gate(want, np.asarray(matrix, dtype=complex), list(targets), nqubits=n)
        device = None if start is None else backend.cast(start, dtype=dtype)
        state = backend.execute_circuit(circuit, initial_state=device).state()
        assert state.dtype == (torch.complex64 if dtype == "complex64" else torch.complex128)
        np.testing.assert_allclose(backend.to_numpy(state), want, atol=10 * PARITY[dtype])
        if start is not None:
            assert state.data_ptr() != device.data_ptr()
            np.testing.assert_array_equal(backend.to_numpy(device), start)


@pytest.mark.parametrize("n", [2, 6])
def test_density_start(backend, dtype, n, rng):
    backend.set_dtype(dtype)
    rho = gm.random_density_matrix(n, rng, dtype)
    circuit = Circuit(n, density_matrix=True)
    circuit.add([gates.SWAP(0, n - 1), gates.H(0)])
    device = backend.cast(rho, dtype=dtype)
    got = backend.to_numpy(backend.execute_circuit(circuit, initial_state=device).state())
    want = er.apply_gate_density_matrix(rho.astype(complex), gm.SWAP, [0, n - 1])
    want = er.apply_gate_density_matrix(want, gm.H, [0])
    np.testing.assert_allclose(got, want, atol=10 * PARITY[dtype])
    np.testing.assert_array_equal(backend.to_numpy(device), rho)


def test_lazily_conjugated_start(backend, rng):
    """A tensor with torch's conjugate bit set is resolved as before."""
    psi = gm.random_state(4, rng)
    lazy = backend.cast(psi).conj()
    circuit = Circuit(4)
    circuit.add(gates.X(1))
    got = backend.execute_circuit(circuit, initial_state=lazy).state()
    want = er.apply_gate(psi.conj(), gm.X, [1], nqubits=4)
    np.testing.assert_allclose(got.resolve_conj().cpu().numpy(), want, atol=1e-13)
