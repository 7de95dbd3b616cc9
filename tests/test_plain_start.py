"""Which initial states a circuit's first pass reads in place."""

import numpy as np
import pytest
import torch

from oracle import einsum_ref as er
from oracle import gate_matrices as gm
from qibojit_amd._qibo import Circuit, gates
from qibojit_amd.backends.hip import HipBackend
from tests.conftest import PARITY


def test_views_off_a_16_byte_boundary_are_copied():
    backend = object.__new__(HipBackend)
    backend._torch_device = torch.device("cpu")
    for dtype in (torch.complex64, torch.complex128):
        buf = torch.zeros(64, dtype=dtype)
        for first in range(4):
            view = buf[first: first + 16]
            assert backend._is_plain_state(view) == (view.data_ptr() % 16 == 0)
    assert not backend._is_plain_state(torch.zeros(64, dtype=torch.complex64)[::2])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [3, 9, 14])
def test_circuit_from_a_view(backend, dtype, n, rng):
    backend.set_dtype(dtype)
    buf = backend.cast(gm.random_state(n + 1, rng, dtype), dtype=dtype)
    start = buf[1: 1 + 2**n]
    psi = backend.to_numpy(start).astype(complex)
    circuit = Circuit(n)
    u = gm.haar_unitary(2 ** min(n, 5), rng)
    targets = tuple(range(min(n, 5)))
    circuit.add([gates.Unitary(u, *targets), gates.H(n - 1)])
    got = backend.to_numpy(backend.execute_circuit(circuit, initial_state=start).state())
    want = er.apply_gate(er.apply_gate(psi, u, list(targets), nqubits=n), gm.H, [n - 1], nqubits=n)
    np.testing.assert_allclose(got, want, rtol=0, atol=PARITY[dtype])
    np.testing.assert_array_equal(backend.to_numpy(start).astype(complex), psi)
