"""Records of a fused circuit go to the library in runs of bounded length,
whatever they come from (no device: the library's call is replaced)."""

import numpy as np
import pytest
import torch

from qibojit_amd._qibo import gates
from qibojit_amd.backends import hip


@pytest.mark.parametrize("kind", ["named", "dense", "channel", "fanout"])
def test_runs_are_bounded(monkeypatch, kind):
    backend = object.__new__(hip.HipBackend)
    backend._torch_device = torch.device("cpu")
    runs = []

    def call(name, *args):
        assert name == "qj_run_gates"
        runs.append(args[9])  # words

    monkeypatch.setattr(hip, "call", call)
    monkeypatch.setattr(hip.HipBackend, "_as_state", lambda self, state: state)
    monkeypatch.setattr(hip.HipBackend, "_stream", lambda self: None)
    monkeypatch.setattr(hip.HipBackend, "_custom_matrix_c128", lambda self, gate: np.asarray(gate.parameters[0]))
    make = {
        "named": lambda: gates.H(0),
        "dense": lambda: gates.Unitary(np.array([[0, 1], [1, 0]]), 1),
        "channel": lambda: gates.KrausChannel((0,), [np.eye(2)]),
        "fanout": lambda: gates.FanOut(0, 1),
    }[kind]
    count = 3 * hip._RECORDS_PER_RUN + 5
    state = torch.zeros((4, 4), dtype=torch.complex128)
    backend._apply_gates_fused([make() for _ in range(count)], state, 2)
    assert len(runs) == 4 and len(set(runs[:3])) == 1 and runs[3] * hip._RECORDS_PER_RUN == 5 * runs[0]
