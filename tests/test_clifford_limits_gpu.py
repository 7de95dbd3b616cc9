"""Symbolic measurement at the largest tableaux of the one-launch loop and
just past them, where the per-qubit pass takes over."""

import numpy as np
import pytest
import torch

from qibojit_amd import _native
from qibojit_amd.backends import clifford_operations_hip as ch

pytestmark = pytest.mark.gpu


def _last_supported(n, ms):
    supported = _native.lib().qj_clifford_forms_supported
    return max(m for m in ms if supported(n, m))


def _ghz(n, k):
    """|0...0> with a GHZ state on the first k qubits."""
    state = ch._clifford_pre_execution_reshape(np.vstack([np.eye(2 * n, 2 * n + 1, dtype=np.uint8),
                                                          np.zeros((1, 2 * n + 1), dtype=np.uint8)]))
    state = ch.H(state, 0, n)
    for q in range(1, k):
        state = ch.CNOT(state, 0, q, n)
    return state


@pytest.mark.parametrize("past", [0, 1])
def test_eight_words_of_rows(past, monkeypatch):
    n = 256
    m = _last_supported(n, range(1, 4000)) + past
    rng = np.random.default_rng(m)
    dense = (rng.random((2 * n + 1, 2 * n + 1)) < 0.3).astype(np.uint8)
    dense[n: 2 * n, :: 3] = 0
    tab = ch._clifford_pre_execution_reshape(dense)
    qubits = [int(q) for q in rng.integers(0, n, size=m)]
    got, k = ch.measurement_forms(tab, qubits, n)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    want, kw = ch.measurement_forms(tab, qubits, n)
    assert k == kw
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("past", [0, 1])
def test_all_qubits_of_a_wide_tableau(past):
    supported = _native.lib().qj_clifford_forms_supported
    n = max(n for n in range(6000, 7000) if supported(n, n)) + past
    forms, k = ch.measurement_forms(_ghz(n, 40), range(n), n)
    assert k == 1 and forms.shape == (n, 2)
    assert forms[:40, 1].all() and not forms[40:].any() and not forms[:, 0].any()
