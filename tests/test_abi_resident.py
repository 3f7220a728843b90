"""eafp_resident as the C compiler lays it out against the Python binding's
mirror, as tests/test_abi_layout.py has it for the other structs; and the
argument checks of the two calls around it, which need no GPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

from eafp import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")
def test_layout(tmp_path):
    names = [n for n, _ in _lib.Resident._fields_]
    src, exe = tmp_path / "layout.c", tmp_path / "layout"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "eafp.h"\nint main(void) {\n'
                   'printf("%zu", sizeof(eafp_resident));\n' +
                   "".join(f'printf(" %zu", offsetof(eafp_resident, {n}));\n' for n in names) + "return 0; }\n")
    subprocess.run(["gcc", "-std=c11", "-Wall", "-I", os.path.join(ROOT, "include"), "-o", str(exe), str(src)],
                   check=True, capture_output=True, timeout=120)
    got = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    assert got == [ctypes.sizeof(_lib.Resident)] + [getattr(_lib.Resident, n).offset for n in names]


def test_null_handles():
    L, r = _lib.load(), _lib.Resident()
    assert L.eafp_batch_resident(None, 0, ctypes.byref(r)) == _lib.EAFP_ERR_ARG
    assert L.eafp_batch_disturb(None, 0, 0, 0) == _lib.EAFP_ERR_ARG
