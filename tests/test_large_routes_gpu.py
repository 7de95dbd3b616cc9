"""Marginals and permuted first passes at sizes where a workgroup takes more
than one row or tile, against reductions and runs on the device."""

import numpy as np
import pytest
import torch

from qibojit_amd._qibo import Circuit, gates

pytestmark = pytest.mark.gpu


def _random_state(n, dtype):
    gen = torch.Generator(device="cuda").manual_seed(n)
    real = torch.float32 if dtype == "complex64" else torch.float64
    state = torch.complex(*(torch.randn(1 << n, generator=gen, dtype=real, device="cuda") for _ in range(2)))
    return state / torch.linalg.vector_norm(state)


# 8192 workgroups share the rows: 1 row each at 21 qubits, 4 at 23 (fewer than
# the eight that a thread loads at a time), 16 at 25, 32 at 26
@pytest.mark.parametrize("n", [21, 23, 25, 26])
@pytest.mark.parametrize("where", ["high", "low", "mixed", "eleven"])
def test_marginal(backend, dtype, n, where):
    backend.set_dtype(dtype)
    qubits = {"high": [0, 1, 2, 3, 4, 5], "low": [n - 1, n - 2, n - 4, n - 5, n - 7, n - 8],
              "mixed": [n - 1, 3, n // 2, 0, n - 6, 7], "eleven": list(range(1, n, 2))[:11]}[where]
    _check_marginal(backend, dtype, n, qubits)


# eight rows at a time: free bits in the row (the lowest), above it and both, up
# to three of them and more, outcomes in and against the order of the memory
@pytest.mark.parametrize("n", [20, 21])
@pytest.mark.parametrize("free", [[], [0], [19], [1, 18], [0, 1, 2], [17, 18, 19], [16, 17, 18, 19], [2, 9, 12, 16, 19]])
@pytest.mark.parametrize("order", ["sorted", "reversed", "shuffled"])
def test_nearly_all_measured(backend, dtype, n, free, order, rng):
    backend.set_dtype(dtype)
    qubits = [q for q in range(n) if q not in free]
    if order == "reversed":
        qubits.reverse()
    elif order == "shuffled":
        qubits = [int(q) for q in rng.permutation(qubits)]
    _check_marginal(backend, dtype, n, qubits)


def _check_marginal(backend, dtype, n, qubits):
    state = _random_state(n, dtype)
    got = backend.calculate_probabilities(state, qubits, n).double()
    probs = torch.view_as_real(state).double().square().sum(-1)
    rest = [q for q in range(n) if q not in qubits]
    order = torch.zeros(1 << n, dtype=torch.int64, device="cuda")  # outcome bits first, the rest below
    index = torch.arange(1 << n, device="cuda")
    for place, q in enumerate(reversed(qubits + rest)):
        order |= ((index >> place) & 1) << (n - 1 - q)
    want = probs[order].reshape(1 << len(qubits), -1).sum(1)
    # FP64 sums of positive terms: at most 32 rows, 9 levels of a tree, 32 + 8 partials
    # of a value; float32 results are rounded once
    rtol = 1.2e-7 if dtype == "complex64" else 3e-14
    np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), rtol=rtol, atol=0)


@pytest.mark.parametrize("n", [22, 23, 25])
@pytest.mark.parametrize("last", ["all", "outer"])
def test_permuted_first_pass(backend, dtype, n, last):
    """A QFT whose last swaps are read out of its start, against the same
    gates in place (a swap pass of their own)."""
    backend.set_dtype(dtype)
    circuit = Circuit(n)
    for q in range(n):
        circuit.add(gates.H(q))
        circuit.add([gates.CU1(p, q, np.pi / 2 ** (p - q)) for p in range(q + 1, n)])
    pairs = n // 2 if last == "all" else 8  # 16 bits, 8 of them above the tile's low run
    circuit.add([gates.SWAP(q, n - 1 - q) for q in range(pairs)])
    start = _random_state(n, dtype)
    got = backend.execute_circuit(circuit, initial_state=start).state()
    want = backend.apply_gates_fused(circuit.queue, start.clone(), n)
    # amplitudes of about 2^-n/2 after at most n roundings each; a misplaced one
    # is off by about 2^-n/2 (2e-4 at 25 qubits)
    atol = 1e-6 if dtype == "complex64" else 1e-13
    assert float((got - want).abs().max()) <= atol
