"""Entry points that several threads may call at once, as far as a machine without a GPU can run them."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# The first launches of a process, all at once: every one finds its kernel, and is refused only because its side holds nothing.
FIRST_LAUNCHES = """
import ctypes as C, sys, threading
from bfuse_project_amd import _lib, operation
l = _lib.lib()
kernels = [k for k in operation.list_kernels() if k.kind == 0]
args = []
for k in kernels:
    a = _lib.LaunchArgsC(mode=operation.MODES["kernel1"], func_a=k.func)
    a.grid_a[:], a.block_a[:] = k.grid, k.block
    args.append(a)
start, said = threading.Barrier(8), []
def work(i):
    start.wait()
    for a in args[i::8]:
        if l.bfuse_launch_packed(C.byref(a)) != -3:          # BFUSE_ERR_STATE
            said.append(l.bfuse_last_error().decode())
threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
[t.start() for t in threads]
[t.join() for t in threads]
sys.exit("\\n".join(said[:5]) or 0)
"""


@pytest.mark.parametrize("attempt", range(5))
def test_first_launches_of_eight_threads(attempt):
    r = subprocess.run([sys.executable, "-c", FIRST_LAUNCHES], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
