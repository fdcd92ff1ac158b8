"""Queued gates against the oracle where planning may merge or exchange them:
CZ pairs that come twice in a run, in either order of their wires, and
operators that are not unitary, which no expectation value queued with them may
pass. Every circuit runs twice, the second time with its kernels compiled."""
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


@pytest.mark.parametrize("bits,tol", [(128, 1e-11), (64, 2e-4)])
@pytest.mark.parametrize("n", [10, 12, 14, 16])
def test_expectations_wait_for_operators_that_are_not_unitary(n, bits, tol):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    from oracle import lq_oracle as O
    C = W.CircuitOp
    rng = np.random.default_rng([n, bits, 7])
    wide = np.eye(8) * 0.9 + 0.1 * np.exp(2j * math.pi * rng.random((8, 8)))
    for matrix, wires in ((np.diag([0.5, 1.3j]), [1]), (np.array([[0.7, 0.4], [-0.2j, 1.1]]), [n - 1]),
                          (np.diag([1.0, 0.6, 0.8j, 1.2]), [2, 5]), (wide, [0, 3, 4])):
        ops = []
        for w in range(n):
            ops += [C("RX", [w], [float(rng.uniform(0, 6.28))]), C("RZ", [w], [float(rng.uniform(0, 6.28))])]
        ops += [C("CNOT", [w, w + 1]) for w in range(n - 1)]
        ops += [C("RY", [w], [float(rng.uniform(0, 6.28))]) for w in range(n)]
        # last, on wires that most of the expectation values do not touch
        ops.append(C("QubitUnitary", wires, [], matrix=matrix.astype(np.complex128)))
        psi = oracle_run(n, ops)
        norm = float(np.vdot(psi, psi).real)
        names = [("PauliZ", "PauliX", "PauliY", "Hadamard")[w % 4] for w in range(n)]
        exp = [O.expval_named(psi, n, names[w], [w]) for w in range(n)]
        xx = ("H", [1.0] * (n - 1), [("T", [("PauliX", w), ("PauliX", w + 1)]) for w in range(n - 1)])
        words = [[("PauliX", w), ("PauliX", w + 1)] for w in range(n - 1)]
        sv = getattr(L, f"StateVectorC{bits}")(n)
        m = getattr(L, f"MeasurementsC{bits}")(sv)
        for _ in range(2):
            # the gates are still queued when the values are asked for
            sv.resetStateVector()
            W.apply_circuit(sv, ops)
            np.testing.assert_allclose(m.expval_named_batch(names, list(range(n))), exp, rtol=0, atol=tol * norm)
            sv.resetStateVector()
            W.apply_circuit(sv, ops)
            got = m.expval(W.hamiltonian_obs([1.0] * (n - 1), words, bits))
            assert abs(got - O.expval_obs(psi, n, xx)) < tol * norm * n
            L.jit_wait()
