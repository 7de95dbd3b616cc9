"""Small tableaux measured on two streams at a time: each call has its own
work space."""

import numpy as np
import pytest
import torch

from qibojit_amd import _native
from qibojit_amd._native import i32_array
from qibojit_amd.backends import clifford_operations_hip as ch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [60, 200, 500])
def test_two_streams(n):
    rng = np.random.default_rng(n)
    qubits = rng.permutation(n)
    ptr, _keep, m = i32_array([int(q) for q in qubits])
    tabs, outs = [], []
    for _ in range(2):
        dense = (rng.random((2 * n + 1, 2 * n + 1)) < 0.3).astype(np.uint8)
        dense[n: 2 * n, :: 3] = 0
        tabs.append(ch._clifford_pre_execution_reshape(dense))
    draws = torch.from_numpy(rng.integers(0, 2, size=m).astype(np.uint8)).cuda()

    def measure(tab, out):
        _native.call("qj_clifford_measure", ch._ptr(tab), n, ptr, m, ch._ptr(draws), 0, ch._ptr(out), ch._ptr(out[m:]),
                     ch._stream(tab))

    for tab in tabs:  # one at a time
        want, out = tab.clone(), torch.zeros(m + 1, dtype=torch.int32, device="cuda")
        measure(want, out)
        outs.append((want, out))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in tabs]
    runs = []
    for _ in range(8):
        for which, stream in enumerate(streams):
            tab, out = tabs[which].clone(), torch.zeros(m + 1, dtype=torch.int32, device="cuda")
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                measure(tab, out)
            runs.append((which, tab, out))
    torch.cuda.synchronize()
    for which, tab, out in runs:
        assert torch.equal(out, outs[which][1]) and torch.equal(tab, outs[which][0])
