"""Host memory that runs out while a gate list is planned: an exception, as from
planning in Python, not the end of the process."""

import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import ctypes, resource
import numpy as np
from qibojit_amd import _native
count = 4096  # five-target matrices of 16 KiB
words = np.tile(np.array([0, 5, 0, 0, 1, 2, 3, 4], dtype=np.int32), count)
params = np.ones(count * 2048)
def run():
    _native.call("qj_run_gates", None, 1, None, _native.QJ_COMPLEX128, 12, 0, 5, 7, words.ctypes.data, len(words),
                 params.ctypes.data, len(params), None, None)
run()
with open("/proc/self/statm") as f:
    used = int(f.read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (16 << 20), resource.RLIM_INFINITY))
try:
    run()
except MemoryError as error:
    print("MemoryError", error)
"""


def test_planner_out_of_memory():
    proc = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr[-500:]
    assert proc.stdout.startswith("MemoryError run_gates")
