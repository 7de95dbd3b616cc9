"""The gate-list planner on the CPU: tests/native/circuit_plan_check.cpp runs
random gate lists through qj_run_gates, whose passes are carried out on host
memory by their documented semantics, and compares with the gates one by one
(no GPU needed)."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(shutil.which(HIPCC) is None and not os.path.exists(HIPCC), reason="hipcc not available")
def test_planned_passes_equal_the_gates_in_order(tmp_path):
    exe = tmp_path / "circuit_plan_check"
    src = os.path.join(HERE, "native", "circuit_plan_check.cpp")
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", src, "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    lines = proc.stdout.strip().splitlines()
    assert proc.returncode == 0, "\n".join(line for line in lines if not line.startswith("ok "))[-2000:]
    assert len(lines) == 8 * 3 * 3 * 7 + 5
    assert sum("permuted=1" in line for line in lines) > 20  # starts read permuted among them
