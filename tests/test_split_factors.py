"""Factors of split 2x2 gates on the CPU: no further from the gate and from norm
one than the factors by angles, and no phase lost that is more than one rounding
(tests/jit_emu/split_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "pennylane-lightning_amd")
LIB = os.path.join(PKG, "lightning_amd", "_lib")


def test_split_factors(tmp_path):
    if not os.path.exists(os.path.join(LIB, "liblq_amd.so")):
        pytest.skip("liblq_amd.so not built")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no host compiler")
    obj, exe = str(tmp_path / "sc.o"), str(tmp_path / "sc")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"),
                    "-c", os.path.join(ROOT, "tests", "jit_emu", "split_check.cpp"), "-o", obj], check=True,
                   capture_output=True)
    subprocess.run([hipcc, obj, "-L", LIB, "-llq_amd", f"-Wl,-rpath,{LIB}", "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]
