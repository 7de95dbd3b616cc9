"""TFIM energies from LDS tiles: passes, rows, selections and few columns."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import einsum_ref as er
from qibojit_amd import _native

pytestmark = pytest.mark.gpu

# (qubits, rows, columns): one pass and many rows, fewer tiles than columns,
# a last pass of one bit and of a full tile, columns that the passes split unevenly
CASES = {
    "complex64": [(13, 64, 32), (14, 33, 7), (19, 1, 64), (22, 1, 5), (23, 1, 1024)],
    "complex128": [(12, 64, 16), (13, 35, 3), (18, 1, 64), (20, 1, 1024), (21, 1, 7)],
}


@pytest.mark.parametrize("ladder", [0, 1])
@pytest.mark.parametrize("case", range(5))
def test_tile_energies(backend, dtype, case, ladder):
    n, rows, ncols = CASES[dtype][case]
    rng = np.random.default_rng(100 * n + ladder)
    stride = (1 << n) + 4
    host = (rng.standard_normal((rows + 1, stride)) + 1j * rng.standard_normal((rows + 1, stride))).astype(dtype)
    host /= np.sqrt(2.0 * (1 << n))
    psi = torch.from_numpy(host).cuda()
    order = rng.permutation(rows + 1)[:rows].astype(np.int32)
    sel = torch.from_numpy(order).cuda()
    partials = torch.full((rows, ncols), np.nan, dtype=torch.float64, device="cuda")
    code = _native.QJ_COMPLEX64 if dtype == "complex64" else _native.QJ_COMPLEX128
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _native.call("qj_tfim_batch", ptr(psi), None, code, n, stride, ptr(sel), rows, 0.7, ladder, ptr(partials), ncols,
                 None)
    got = partials.sum(dim=1).cpu().numpy()
    k = np.arange(1 << n)
    for b in sorted({0, rows - 1, rows // 2}):
        state = host[order[b], : 1 << n].astype(np.complex128)
        # the ladder maps amplitude k ^ (k >> 1) to k
        want = er.tfim_energy(state[k ^ (k >> 1)] if ladder else state, 0.7)
        # FP64 sums of products of the stored amplitudes, |terms| summing to about n
        assert abs(got[b] - want) < 1e-11 * n, (n, b)
