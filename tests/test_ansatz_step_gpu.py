"""Steps of many circuits in one launch against one register pass per bit,
equal to the last digit, and the planner of the steps."""

import ctypes

import numpy as np
import pytest
import torch

from qibojit_amd import _native
from qibojit_amd._native import call, i32_array
from qibojit_amd.ansatz import LOAD_LADDER, LOAD_PLAIN, LOAD_ZERO, register_passes
from qibojit_amd.batch import AnsatzBatch, step_passes


@pytest.mark.parametrize("run", [3, 4])
@pytest.mark.parametrize("k", [1, 3, 4, 5])
@pytest.mark.parametrize("n", [12, 13, 14, 20, 21, 27, 31])
def test_steps_keep_the_order_and_whole_lines(n, k, run):
    steps = step_passes(n, k, run)
    assert [b for ps in steps for b in ps.bits] == [b for ps in register_passes(n, k) for b in ps.bits]
    for ps in steps:
        fill = [b for b in range(n) if b not in ps.bits][: 12 - len(ps.bits)]
        assert 1 <= len(ps.bits) <= 10 and set(range(run)) <= set(ps.bits) | set(fill)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _rows(rows):
    return np.array([r + [0] * (19 - len(r)) for r in rows], dtype=np.int64)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["complex64", "complex128"])
@pytest.mark.parametrize("load", [LOAD_ZERO, LOAD_PLAIN, LOAD_LADDER])
@pytest.mark.parametrize("bits", [[0], [11, 3, 0], [0, 3, 6, 9, 1], [0, 4, 8, 11, 1, 5], [2, 5, 8, 11, 0, 3, 6, 9, 1, 4],
                                  [13, 12, 10, 7, 1, 2, 3, 4, 5, 6]])
def test_step_equals_register_passes(prec, load, bits):
    n, count = 14 if max(bits) > 11 else 12, 3
    tdtype = getattr(torch, prec)
    code = _native.QJ_COMPLEX64 if prec == "complex64" else _native.QJ_COMPLEX128
    rng = np.random.default_rng(len(bits))
    u = len(bits)
    mats = torch.from_numpy(rng.normal(size=(count, u, 4)) + 1j * rng.normal(size=(count, u, 4))).to(tdtype).cuda()
    start = torch.from_numpy(rng.normal(size=(count, 1 << n)) + 1j * rng.normal(size=(count, 1 << n))).to(tdtype).cuda()
    want = torch.empty_like(start)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    eye = torch.eye(2, dtype=tdtype, device="cuda").reshape(1, 1, 4).expand(count, 1, 4)
    for i, bit in enumerate(bits):  # a register pass of two bits, the other one left as it is
        other = bit + 1 if bit + 1 < n else bit - 1
        parts = [mats[:, i: i + 1], eye]
        part = torch.cat(parts if bit < other else parts[::-1], dim=1).contiguous()
        ptr, _keep, nbits = i32_array(sorted((bit, other)))
        call("qj_rot_pass", None if i == 0 and load == LOAD_ZERO else _p(want if i else start), _p(want), None, None,
             code, n, 1 << n, None, count, ptr, nbits, 1, None, LOAD_PLAIN if i else load, _p(part), 4 * nbits, None, 4,
             stream)
    half = count << n
    pool = torch.zeros(2 * half + (2 << 12), dtype=tdtype, device="cuda")
    pool[:half] = start.reshape(-1)
    in_place = load == LOAD_PLAIN
    ka = min(5, u)
    rows = _rows([[n, count, -1 if load == LOAD_ZERO else 0, 0 if in_place else half, int(load == LOAD_LADDER), 0, u, ka,
                   u - ka, *bits],
                  [12, 1, -1, 2 * half + (1 << 12), 0, 0, u, 1, 0, 0]])
    call("qj_ansatz_step", _p(pool), code, pool.numel(), _p(mats), mats.numel(), ctypes.c_void_p(rows.ctypes.data), 2,
         stream)
    got = pool[:half] if in_place else pool[half: 2 * half]
    assert torch.equal(got.view(count, -1), want)
    last = pool[2 * half:].cpu()
    assert torch.equal(last[: 1 << 12], torch.zeros(1 << 12, dtype=tdtype))
    assert torch.equal(last[1 << 12: (1 << 12) + 2], mats[0, 0, [0, 2]].cpu()) and not last[(1 << 12) + 2:].any()


@pytest.mark.gpu
def test_step_refuses_what_does_not_fit():
    pool = torch.zeros(2 << 12, dtype=torch.complex64, device="cuda")
    mats = torch.zeros((4, 4), dtype=torch.complex64, device="cuda")
    good = [12, 1, 0, 4096, 1, 0, 2, 2, 0, 0, 1]
    for i, value in ((0, 11), (1, 2), (2, 4097), (2, 4096), (3, 4100), (5, 3), (7, 0), (8, 6), (9, 12), (10, 0)):
        row = list(good)
        row[i] = value
        with pytest.raises(Exception):
            call("qj_ansatz_step", _p(pool), _native.QJ_COMPLEX64, pool.numel(), _p(mats), mats.numel(),
                 ctypes.c_void_p(_rows([row]).ctypes.data), 1, None)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["complex64", "complex128"])
def test_batch_of_uneven_depths(prec):
    shapes = [(14, 1), (15, 4), (14, 5), (12, 2), (13, 3), (21, 2), (14, 2), (15, 1)]
    rng = np.random.default_rng(3)
    params = [rng.uniform(-3, 3, 2 * n * nl) for n, nl in shapes]
    batch = AnsatzBatch(shapes, dtype=prec, plan={n: ("pass", 5) for n, _ in shapes})
    batch.set_parameters(params)
    batch.run()
    got = batch.energies().cpu().numpy()
    for (n, nl), p, e in zip(shapes, params, got):
        one = AnsatzBatch([(n, nl)], dtype="complex128", plan={n: ("pass", 4)})
        one.set_parameters([p])
        one.run()
        np.testing.assert_allclose(e, one.energies().item(), rtol=0, atol=n * (2e-5 if prec == "complex64" else 1e-12))
