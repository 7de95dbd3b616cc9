"""Channels as superoperators on the row and column bits of rho."""

import numpy as np
import pytest

from oracle import einsum_ref as er
from oracle import gate_matrices as gm
from qibojit_amd._qibo import Circuit, gates
from qibojit_amd.backends.matrices import KernelMatrices
from qibojit_amd.fusion import channel_superoperator
from tests.conftest import ATOL


def _damping(gamma):
    return [np.diag([1, np.sqrt(1 - gamma)]), np.array([[0, np.sqrt(gamma)], [0, 0]])]


def _channels(n, rng):
    """(channel, reference map) pairs of every route: one qubit, two qubits
    (in both orders and as single-qubit terms), and three (the operator sum)."""
    paulis = [gm.X, gm.Y, gm.Z]
    u4 = gm.haar_unitary(4, rng)
    top, low, mid = 0, n - 1, n // 2
    cases = [
        ([(0.1, (low,), paulis[0]), (0.2, (low,), paulis[1]), (0.05, (low,), paulis[2])], True),
        ([(1.0, (top,), k) for k in _damping(0.3)], False),
    ]
    if n >= 2:
        cases.append(([(0.3, (low, top), u4), (0.1, (top, low), gm.SWAP)], True))
        cases.append(([(0.2, (top,), gm.Y), (0.4, (low,), gm.haar_unitary(2, rng))], True))
        cases.append(([(1.0, (top, low), np.kron(a, b)) for a in _damping(0.2) for b in _damping(0.6)], False))
    if n >= 3:
        cases.append(([(0.25, (low,), gm.X), (0.5, (mid, top), u4)], True))
    for terms, unitary in cases:
        if unitary:
            channel = gates.UnitaryChannel([q for _, q, _ in terms], [(p, m) for p, _, m in terms])
        else:
            channel = gates.KrausChannel([q for _, q, _ in terms], [m for _, _, m in terms])
        yield channel, terms, unitary


def _reference(rho, terms, unitary):
    new = (1 - sum(p for p, _, _ in terms)) * rho if unitary else 0 * rho
    for p, qubits, m in terms:
        new = new + p * er.apply_gate_density_matrix(rho, np.asarray(m, dtype=complex), list(qubits))
    return new


def test_superoperator_matches_operator_sum(rng):
    encode = KernelMatrices("complex128").encode
    rho = gm.random_density_matrix(2, rng)
    vec = rho.reshape(-1)  # row bits, then column bits
    for channel, terms, unitary in _channels(2, rng):
        block = sorted({q for _, qs, _ in terms for q in qs})
        s = channel_superoperator(encode, channel, block)
        full = er.apply_gate(vec, s, block + [q + 2 for q in block], nqubits=4)
        np.testing.assert_allclose(full.reshape(4, 4), _reference(rho, terms, unitary), atol=1e-14)


def test_singular_unitary_term_is_refused():
    channel = gates.UnitaryChannel([(0,)], [(0.5, np.diag([1.0, 0.0]))])
    with pytest.raises(np.linalg.LinAlgError):
        channel_superoperator(KernelMatrices("complex128").encode, channel, [0])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 5, 7])
def test_channels_against_einsum(backend, dtype, n, rng):
    backend.set_dtype(dtype)
    rho = gm.random_density_matrix(n, rng, dtype)
    for channel, terms, unitary in _channels(n, rng):
        want = _reference(rho.astype(complex), terms, unitary)
        device = backend.cast(rho, dtype=dtype, copy=True)
        got = backend.to_numpy(backend.apply_channel(channel, device, n))
        np.testing.assert_allclose(got, want, atol=ATOL[dtype])
        circuit = Circuit(n, density_matrix=True)
        circuit.add([gates.H(0), channel, gates.RY(n - 1, 0.3)])
        got = backend.to_numpy(backend.execute_circuit(circuit, initial_state=rho).state())
        want = er.apply_gate_density_matrix(rho.astype(complex), gm.H, [0])
        want = er.apply_gate_density_matrix(_reference(want, terms, unitary), gm.RY(0.3), [n - 1])
        np.testing.assert_allclose(got, want, atol=ATOL[dtype])
