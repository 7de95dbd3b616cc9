"""Marginals over more than five qubits (row kernel) and the sequential CDF
of the shot sampler at the edges of its chunks."""

import numpy as np
import pytest
import torch

from oracle import einsum_ref as er
from oracle import gate_matrices as gm

pytestmark = pytest.mark.gpu

# (qubits of the state, measured qubits): everything measured, rows larger
# than the state, only bits above the row, only bits inside it, both in an
# unsorted order, one chunk per outcome and many
CASES = [
    (6, (0, 1, 2, 3, 4, 5)),
    (7, (6, 0, 3, 1, 5, 2)),
    (8, (7, 6, 5, 4, 3, 2, 1, 0)),
    (9, (8, 0, 7, 1, 6, 2)),
    (10, (9, 8, 7, 6, 5, 4, 3, 2, 1, 0)),
    (13, (0, 1, 2, 3, 4, 5)),
    (13, (12, 11, 10, 9, 8, 7)),
    (14, (13, 0, 7, 4, 9, 2, 5)),
    (19, (3, 0, 2, 1, 4, 5)),
    (20, (19, 2, 11, 5, 18, 7, 0, 12, 13)),
]


@pytest.mark.parametrize("nqubits,qubits", CASES)
def test_wide_marginals(backend, dtype, nqubits, qubits, rng):
    backend.set_dtype(dtype)
    state = gm.random_state(nqubits, rng, dtype)
    got = backend.to_numpy(backend.calculate_probabilities(backend.cast(state, dtype=dtype), qubits, nqubits))
    want = er.probabilities(state.astype(complex), list(qubits))
    # FP64 sums of at most 2^n terms in a tree, rounded once to the result's type
    eps = 1.2e-7 if dtype == "complex64" else 1e-14
    np.testing.assert_allclose(got, want.reshape(-1), rtol=eps, atol=1e-16)


@pytest.mark.parametrize("nqubits,qubits", [c for c in CASES if c[0] <= 9])
def test_wide_density_marginals(backend, dtype, nqubits, qubits, rng):
    backend.set_dtype(dtype)
    rho = gm.random_density_matrix(nqubits, rng, dtype)
    got = backend.to_numpy(backend.calculate_probabilities(backend.cast(rho, dtype=dtype), qubits, nqubits))
    want = er.probabilities_density_matrix(rho.astype(complex), list(qubits))
    eps = 1.2e-7 if dtype == "complex64" else 1e-14
    np.testing.assert_allclose(got, want.reshape(-1), rtol=eps, atol=1e-16)


def test_wide_marginal_of_a_view(backend, rng):
    """A complex64 state that starts 8 bytes off a 16-byte boundary."""
    backend.set_dtype("complex64")
    n, qubits = 12, (11, 3, 0, 7, 5, 9)
    buf = backend.cast(gm.random_state(n + 1, rng, "complex64"), dtype="complex64")
    state = buf[1: 1 + 2**n]
    got = backend.to_numpy(backend.calculate_probabilities(state, qubits, n))
    want = er.probabilities(backend.to_numpy(state).astype(complex), list(qubits))
    np.testing.assert_allclose(got, want.reshape(-1), rtol=1.2e-7, atol=1e-16)


@pytest.mark.parametrize("nstates", [15, 16, 17, 2047, 2048, 2049, 4095, 6145])
def test_sequential_cdf_matches_numpy_choice(backend, nstates):
    probs = np.random.default_rng(nstates).random(nstates)
    probs /= probs.sum()
    backend.set_seed(nstates)
    got = backend.to_numpy(backend.sample_shots(torch.from_numpy(probs).cuda(), 20000))
    np.testing.assert_array_equal(got, np.random.RandomState(nstates).choice(nstates, 20000, p=probs))
