"""Ansatz matrices built on the device against the host's RY and RZ."""

import numpy as np
import pytest

from qibojit_amd.ansatz import AnsatzEngine, HardwareEfficientAnsatz
from qibojit_amd.batch import AnsatzBatch, _fused_layers

pytestmark = pytest.mark.gpu


def _ulp(prec):
    return 2.0 ** -23 if prec == "complex64" else 2.0 ** -50


@pytest.mark.parametrize("prec", ["complex64", "complex128"])
@pytest.mark.parametrize("n,layers,batch", [(2, 1, 1), (5, 3, 2), (13, 2, 3), (14, 33, 1)])
def test_engine_matrices(n, layers, batch, prec):
    eng = AnsatzEngine(HardwareEfficientAnsatz(n, layers), batch=batch, dtype=prec, device="cuda")
    p = np.random.default_rng(n).uniform(-7, 7, (batch, 2 * n * layers))
    for passes, width, steps, host in (
        (eng.passes_f, eng.width_f, 1, eng._forward_mats(p)),
        (eng.passes_a, eng.width_a, 2, eng._adjoint_mats(p)),
    ):
        got = eng._device_mats(p, passes, width, steps).cpu().numpy()
        want = host.cpu().numpy()
        assert got.shape == want.shape
        np.testing.assert_allclose(got, want, rtol=0, atol=_ulp(prec))


@pytest.mark.parametrize("prec", ["complex64", "complex128"])
def test_batch_matrices(prec):
    shapes = [(3, 2), (14, 1), (2, 1), (14, 3), (15, 2), (3, 4)]
    rng = np.random.default_rng(5)
    params = [rng.uniform(-7, 7, 2 * n * nl) for n, nl in shapes]
    eng = AnsatzBatch(shapes, dtype=prec, device="cuda")
    eng.set_parameters(params)
    flat = eng.lds_mats.cpu().numpy().reshape(-1, 4)
    at = 0
    for c in eng.order[: eng.nlds]:
        n, nl = shapes[c]
        np.testing.assert_allclose(flat[at: at + n * nl], _fused_layers(n, nl, params[c]).reshape(-1, 4),
                                   rtol=0, atol=_ulp(prec))
        at += n * nl
    for grp in eng.pass_groups:
        mats = grp.mats.cpu().numpy()
        want = np.zeros_like(mats)
        for s, c in enumerate(grp.members):
            m = _fused_layers(grp.n, shapes[c][1], params[c])
            for i, ps in enumerate(grp.passes):
                for a, bit in enumerate(ps.bits):
                    if bit in ps.rot:
                        want[: m.shape[0], i, s, a, 0] = m[:, bit]
        np.testing.assert_allclose(mats, want, rtol=0, atol=_ulp(prec))
