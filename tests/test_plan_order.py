"""The order in which plans run their ops, on the CPU: random programs of gates
and dots are planned by liblq_amd.so's planner, interpreted pass by pass on the
host and compared, states and dots, with the ops applied one after the other
(tests/jit_emu/plan_order_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "pennylane-lightning_amd")
LIB = os.path.join(PKG, "lightning_amd", "_lib")


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    if not os.path.exists(os.path.join(LIB, "liblq_amd.so")):
        pytest.skip("liblq_amd.so not built")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan_order")
    obj, exe = str(d / "poc.o"), str(d / "poc")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"),
                    "-c", os.path.join(ROOT, "tests", "jit_emu", "plan_order_check.cpp"), "-o", obj], check=True,
                   capture_output=True)
    subprocess.run([hipcc, obj, "-L", LIB, "-llq_amd", f"-Wl,-rpath,{LIB}", "-o", exe], check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("family,seeds", [("words", 500), ("cz", 200), ("nonunitary", 200), ("partial", 200), ("long", 1)])
def test_plans_keep_the_order_of_their_ops(compiled, family, seeds):
    r = subprocess.run([compiled, family, str(seeds)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]
    assert f"{4 * seeds} plans, 0 wrong" in r.stdout
