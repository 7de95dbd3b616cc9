"""Few measured qubits of a wide tableau: on both sides of the line between the
one-launch loop and the launches per qubit, and where a single workgroup writes
the tableau itself, against the per-qubit entry points."""

import numpy as np
import pytest
import torch

from qibojit_amd.backends import clifford_operations_hip as ch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (31, 2), (32, 1), (128, 3), (129, 3), (257, 1), (257, 2), (2499, 2), (2500, 2),
                                 (2501, 3), (5001, 3), (5001, 4)])
def test_few_measured_qubits(n, m):
    rng = np.random.default_rng(n + m)
    dense = (rng.random((2 * n + 1, 2 * n + 1)) < 0.3).astype(np.uint8)
    dense[n: 2 * n, :: 3] = 0  # determined outcomes
    tab = ch._clifford_pre_execution_reshape(dense)
    qubits = [int(q) for q in rng.integers(0, n, size=m)]
    want = tab.clone()
    np.random.seed(n)
    outcomes = []
    for q in qubits:
        p = ch.first_stabilizer(want, q, n)
        outcomes.append(int((ch._random_outcome(want, [p], q, n) if p >= 0 else ch._determined_outcome(want, q, n))[1]))
    np.random.seed(n)
    assert ch.M(tab, qubits, n, collapse=True) == outcomes
    assert torch.equal(tab, want)
