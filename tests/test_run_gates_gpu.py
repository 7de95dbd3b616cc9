"""Gate lists planned by the library: every named gate, dense and diagonal
blocks, swaps and controls in random order, against the einsum closed form
gate by gate."""

import ctypes

import numpy as np
import pytest

from oracle import einsum_ref as er
from oracle import gate_matrices as gm
from oracle import port
from qibojit_amd import _native
from qibojit_amd._qibo import Circuit, gates
from qibojit_amd.fusion import target_block
from qibojit_amd.records import GATE_CODES, Records
from tests.conftest import PARITY

THREE = {"TOFFOLI": 3, "CCZ": 3}


def _named(name, q, rng):
    cls = getattr(gates, name)
    nq = THREE.get(name, 2 if name.startswith("C") else 1)
    return cls(*q[:nq], *[float(x) for x in rng.uniform(-7, 7, GATE_CODES[name][1])]), nq


def random_gates(n, count, rng, kmax=5):
    """A shuffled mixture of every record form that n qubits allow."""
    out = []
    names = sorted(GATE_CODES)
    while len(out) < count:
        q = [int(x) for x in rng.permutation(n)]
        pick = rng.integers(10)
        if pick < 5:
            name = names[rng.integers(len(names))]
            if THREE.get(name, 2 if name.startswith("C") else 1) > n:
                continue
            gate, used = _named(name, q, rng)
            if pick == 0 and used + 1 <= n:
                gate = gate.controlled_by(*q[used: min(n, used + 2)])
            out.append(gate)
        elif pick == 5 and n >= 2:
            out.append(gates.SWAP(q[0], q[1]))
        elif pick == 6 and n >= 4:  # a run of swaps on distinct qubits
            out += [gates.SWAP(q[2 * j], q[2 * j + 1]) for j in range(n // 2)]
        elif pick == 7:
            k = int(rng.integers(1, min(n, kmax) + 1))
            out.append(gates.Unitary(gm.haar_unitary(2**k, rng), *q[:k]))
        elif pick == 8:
            out.append(gates.Unitary(np.diag(np.exp(1j * rng.uniform(-3, 3, 2))), q[0]))
        elif n >= 2:
            out.append([gates.fSim(q[0], q[1], 0.3, -0.8), gates.RX(q[0], np.array(0.7)), gates.I(q[0], q[1]),
                        gates.RZZ(q[0], q[1], 0.4)][rng.integers(4)])
    return out


def _apply(state, gate, n):
    """The gate on a complex128 host vector, by the port's gate encodings
    where it has them, else by the textbook matrix over all its qubits."""
    if type(gate).__name__ in ("I", "RZZ"):
        return er.apply_gate(state, gate.matrix(), list(gate.target_qubits), nqubits=n)
    return er.apply_gate(state, target_block(port.custom_matrix, gate), list(gate.target_qubits),
                         list(gate.control_qubits), nqubits=n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 8, 9, 10, 12, 13, 14, 16])
@pytest.mark.parametrize("seed", [0, 1])
def test_lists_against_port(backend, dtype, n, seed):
    backend.set_dtype(dtype)
    rng = np.random.default_rng(1000 * n + seed)
    circuit = Circuit(n)
    circuit.add(random_gates(n, 60, rng))
    psi = gm.random_state(n, rng, dtype)
    want = psi.astype(complex)
    for gate in circuit.queue:
        want = _apply(want, gate, n)
    got = backend.to_numpy(backend.execute_circuit(circuit, initial_state=backend.cast(psi, dtype=dtype)).state())
    np.testing.assert_allclose(got, want, atol=20 * PARITY[dtype], rtol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7])
def test_density_lists_against_einsum(backend, dtype, n, rng):
    backend.set_dtype(dtype)
    circuit = Circuit(n, density_matrix=True)
    circuit.add(random_gates(n, 30, rng, kmax=4))
    rho = gm.random_density_matrix(n, rng, dtype)
    want = rho.astype(complex)
    for gate in circuit.queue:
        # U rho, then (U (U rho)^+)^+
        half = np.stack([_apply(col, gate, n) for col in want.T], axis=1)
        want = np.stack([_apply(row, gate, n) for row in half.conj()], axis=0).conj()
    got = backend.to_numpy(backend.execute_circuit(circuit, initial_state=backend.cast(rho, dtype=dtype)).state())
    np.testing.assert_allclose(got, want, atol=20 * PARITY[dtype], rtol=0)


@pytest.mark.gpu
def test_long_list_runs_in_parts(backend, rng):
    """More gates than one run plans, with a wide gate between."""
    n = 11
    circuit = Circuit(n)
    circuit.add(random_gates(n, 700, rng, kmax=3))
    circuit.add(gates.Unitary(gm.haar_unitary(64, rng), *range(6)))
    circuit.add(random_gates(n, 520, rng, kmax=3))
    want = np.zeros(2**n, dtype=complex)
    want[0] = 1
    for gate in circuit.queue:
        want = _apply(want, gate, n)
    got = backend.to_numpy(backend.execute_circuit(circuit).state())
    np.testing.assert_allclose(got, want, atol=1e-11, rtol=0)


def _plan(circuit, n, low, high):
    records = Records()
    for gate in circuit.queue:
        assert records.add(gate, port.custom_matrix)
    passes = ctypes.c_int32(0)
    _native.call("qj_run_gates", None, 0, None, _native.QJ_COMPLEX128, n, 0, low, high,
                 records.words.buffer_info()[0], len(records.words), records.params.buffer_info()[0],
                 len(records.params), ctypes.byref(passes), None)
    return passes.value


def test_planner_collects_commuting_gates():
    """Gates of later layers join a pass that holds their bits: two layers on
    the same high bits need one pass, a disjoint set of bits a second one."""
    n, low, high = 20, 5, 7
    c = Circuit(n)
    for _ in range(2):
        for q in range(n):
            c.add(gates.RY(q, 0.1))
    assert _plan(c, n, low, high) == 3  # 15 high bits, 7 per pass
    c = Circuit(n)
    for q in range(7):
        c.add(gates.H(q))
    c.add(gates.H(10))
    for q in range(7):
        c.add(gates.T(q))
        c.add(gates.H(q))
    assert _plan(c, n, low, high) == 2


@pytest.mark.parametrize("words,params", [
    ([99, 1, 0, 0], []), ([3, 1, 0], []), ([3, 1, 0, 5], []), ([3, 1, 1, 0, 0], []), ([3, 2, 0, 0, 1], []),
    ([2, 2, 1, 0, 1, 2], []), ([13, 1, 0, 0], []), ([0, 1, 0, 0], [1.0] * 7), ([3, 1, -1, 0], []),
])
def test_bad_records_are_refused(words, params):
    w = (ctypes.c_int32 * len(words))(*words)
    p = (ctypes.c_double * max(1, len(params)))(*params)
    with pytest.raises(ValueError):
        _native.call("qj_run_gates", None, 0, None, _native.QJ_COMPLEX128, 4, 0, 4, 0, w, len(words), p, len(params),
                     None, None)
