"""Five-target blocks at the sizes where the launch changes how many column
groups a wave takes."""

import numpy as np
import pytest

from oracle import einsum_ref as er
from oracle import gate_matrices as gm
from qibojit_amd._qibo import gates
from tests.conftest import PARITY

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 10, 15, 18, 20, 21, 22])
@pytest.mark.parametrize("low", [True, False])
def test_five_target_blocks(backend, dtype, n, low, rng):
    backend.set_dtype(dtype)
    u = gm.haar_unitary(32, rng)
    targets = tuple(range(n - 5, n)) if low else (3, 0, n - 5, 1, n - 1)
    psi = gm.random_state(n, rng, dtype)
    got = backend.to_numpy(backend.apply_gate(gates.Unitary(u, *targets), backend.cast(psi, copy=True, dtype=dtype), n))
    want = er.apply_gate(psi.astype(complex), u, list(targets), nqubits=n)
    np.testing.assert_allclose(got, want, atol=PARITY[dtype], rtol=0)
