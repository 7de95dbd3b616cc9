"""Shape of the one-launch Clifford measurement loop: host arithmetic."""

import os
import shutil
import subprocess
import sys

import pytest

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
from qibojit_amd import _native
print([_native.lib().qj_clifford_forms_supported(n, m) for n in (1, 100, 256, 257, 1000, 4000) for m in (1, 100, 1000)])
"""


@pytest.mark.parametrize("value", ["0", "3", "8", "x"])
def test_shape_depends_on_the_tableau_alone(value):
    out = []
    for env in ({}, {"QJ_RT": value}):
        proc = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, env={**os.environ, **env},
                              capture_output=True, text=True, timeout=300)
        assert proc.returncode == 0, proc.stderr[-500:]
        out.append(proc.stdout)
    assert out[0] == out[1]


@pytest.mark.skipif(shutil.which(HIPCC) is None and not os.path.exists(HIPCC), reason="hipcc not available")
def test_accepted_shapes_fit_a_compute_unit(tmp_path):
    """Every accepted tableau, fixed and dynamic LDS together, fits 160 KiB,
    up to the last one that does."""
    exe = tmp_path / "cliff_plan_check"
    src = os.path.join(ROOT, "tests", "native", "cliff_plan_check.cpp")
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", src, "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout[-2000:]
