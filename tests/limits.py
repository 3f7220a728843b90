"""Runs Python in a process of its own whose HIP allocations pass tests/hip_shim.c
(`shim`, a ctypes handle).  The GPU tests of scarce memory use it."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HEAD = '''
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.shim_used.restype = shim.shim_times.restype = shim.shim_calls.restype = ctypes.c_long
for f in (shim.shim_limit, shim.shim_fail, shim.shim_pinned, shim.shim_slow):
    f.argtypes, f.restype = [ctypes.c_long], None
sys.path[:0] = [sys.argv[2], sys.argv[3]]
import numpy as np
import eafp
from eafp import _lib, fields, systems
assert "torch" not in sys.modules
'''


def run(tmp_path, code):
    so = os.path.join(str(tmp_path), "hip_shim.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "hip_shim.c"), "-ldl"],
                   check=True, capture_output=True, timeout=60)
    out = subprocess.run([sys.executable, "-u", "-c", HEAD + code, so, os.path.join(ROOT, "hornofusion-full3d_amd"),
                          HERE], capture_output=True, text=True, timeout=100)
    print(out.stdout, out.stderr, flush=True)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-2000:]
    return out.stdout
