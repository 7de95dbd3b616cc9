"""The one-launch measurement loop (rows in LDS) against the per-qubit entry
points, and its symbolic form against the per-qubit symbolic pass."""

import numpy as np
import pytest
import torch

from qibojit_amd.backends import clifford_operations_hip as ch

pytestmark = pytest.mark.gpu

# one workgroup with 1, 2, 4 and 8 words of rows, several workgroups, rows
# that end inside, at and just past a word
SIZES = [1, 2, 31, 32, 33, 64, 65, 100, 128, 129, 255, 256, 257, 288, 300, 513, 1000]


def _random_tableau(rng, n):
    """Random bits in every row (scratch row included): not a state, so every
    branch of the sign rule and of the scratch row is met."""
    dense = (rng.random((2 * n + 1, 2 * n + 1)) < 0.3).astype(np.uint8)
    dense[n: 2 * n, :: 3] = 0  # columns without a stabilizer: determined outcomes
    return ch._clifford_pre_execution_reshape(dense)


def _per_qubit(tab, qubits, n):
    sample = []
    for q in qubits:
        p = ch.first_stabilizer(tab, q, n)
        if p >= 0:
            _, out = ch._random_outcome(tab, [p], q, n)
        else:
            _, out = ch._determined_outcome(tab, q, n)
        sample.append(int(out))
    return sample


@pytest.mark.parametrize("n", SIZES)
def test_rows_loop_equals_per_qubit_calls(n):
    rng = np.random.default_rng(n)
    tab = _random_tableau(rng, n)
    qubits = [int(v) for v in rng.integers(0, n, size=min(2 * n, 60))]
    ref = tab.clone()
    np.random.seed(n)
    want = _per_qubit(ref, qubits, n)
    np.random.seed(n)
    got = ch.M(tab, qubits, n, collapse=True)
    assert got == want
    assert torch.equal(tab, ref)


@pytest.mark.parametrize("n", SIZES)
def test_forms_equal_the_per_qubit_symbolic_pass(n, monkeypatch):
    rng = np.random.default_rng(n + 1)
    tab = _random_tableau(rng, n)
    before = tab.clone()
    qubits = [int(v) for v in rng.permutation(n)[: min(n, 70)]]
    got, k = ch.measurement_forms(tab, qubits, n)
    assert torch.equal(tab, before)
    # a stream under capture takes the per-qubit pass
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    want, kw = ch.measurement_forms(tab, qubits, n)
    assert k == kw
    np.testing.assert_array_equal(got, want)
