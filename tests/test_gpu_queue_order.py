"""Queued gates against the oracle where planning may merge or exchange them:
CZ pairs that come twice in a run, in either order of their wires. Every
circuit runs twice, the second time with its kernels compiled."""
import math

import numpy as np
import pytest

from helpers import TOL_C128, TOL_C64, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,tol", [(128, TOL_C128), (64, TOL_C64)])
@pytest.mark.parametrize("n", [11, 12, 14, 16])
def test_cz_twice(n, bits, tol):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    rng = np.random.default_rng([n, bits])
    C = W.CircuitOp
    ops = [C("RY", [w], [float(rng.uniform(0.3, 2.8))]) for w in range(n)]
    ops += [C("CZ", [0, 1]), C("CZ", [1, 0])]
    for k in range(40):
        a, b = (int(x) for x in rng.choice(n, size=2, replace=False))
        ops += [C("CZ", [a, b]), C("CZ", [b, a])] if k % 3 == 0 else [C("CZ", [a, b])]
        if k % 5 == 0:
            ops += [C("RZ", [a], [float(rng.uniform(0, 2 * math.pi))]), C("CZ", [b, a]),
                    C("ControlledPhaseShift", [a, b], [0.7])]
    ops += [C("RX", [w], [0.4]) for w in range(n)]
    psi = oracle_run(n, ops)
    sv = getattr(L, f"StateVectorC{bits}")(n)
    for _ in range(2):
        sv.resetStateVector()
        W.apply_circuit(sv, ops)
        np.testing.assert_allclose(sv.state(), psi, rtol=0, atol=tol)
        L.jit_wait()
