"""The parts of an overlapped line-TDMA sweep (csrc/tdma_line.hpp, chain_part):
what each part needs is there when its stream reaches it, on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not available")
def test_tdma_parts(tmp_path):
    exe = tmp_path / "tdma_parts_check"
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "-x", "hip", "--offload-arch=gfx950", "-std=c++17",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-O1", "-g", "-Xarch_host", "-fsanitize=address",
           "-o", str(exe), os.path.join(HERE, "tdma_parts_check.cpp")]
    subprocess.run(cmd, check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok "), out.stdout
