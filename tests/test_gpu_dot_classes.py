"""Dots in specialised passes: generators X, Y, Z and parities with and without
controls on register and thread bits, the parts that are used (imaginary in
the adjoint, real in expectations, both in the vector-Jacobian product), phases
and rotations that move past dots, X and SWAP as exchanges, and operators that
are not unitary, which no dot may change places with. Every circuit runs twice,
the second time with its kernels compiled."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def circuit(n, rng, matrix=None):
    from lightning_amd import workloads as W
    C = W.CircuitOp
    a = lambda: [float(rng.uniform(0, 2 * math.pi))]  # noqa: E731
    ops = []
    for layer in range(2):
        for w in range(n):
            ops += [C("RZ", [w], a()), C("RY", [w], a()), C("RX", [w], a())]
        for w in range(0, n - 1, 3):
            ops += [C("CNOT", [w, w + 1]), C("CRX", [w + 1, w], a()), C("SWAP", [w, (w + 5) % n]),
                    C("CRZ", [w, (w + 2) % n], a()), C("IsingZZ", [w, (w + 3) % n], a()), C("PauliX", [w]),
                    C("CRY", [(w + 7) % n, w], a()), C("PhaseShift", [w], a()),
                    C("ControlledPhaseShift", [w, (w + 4) % n], a()), C("MultiRZ", [w, (w + 2) % n, (w + 6) % n], a())]
        ops += [C("PauliX", [n - 1], ctrls=[0, n // 2, n - 2], cvals=[1, 0, 1]), C("RY", [1], a(), ctrls=[n - 1], cvals=[0])]
    if matrix is not None:
        ops.insert(len(ops) // 2, C("QubitUnitary", [n - 3], [0.0], matrix=matrix))
    return ops


def oracle_ops(ops):
    from oracle import lq_oracle as O
    return [O.Op(o.name, o.wires, o.params, o.inverse, o.matrix, o.ctrls, o.cvals) for o in ops]


@pytest.mark.parametrize("bits,tol", [(128, 1e-10), (64, 5e-4)])
@pytest.mark.parametrize("n", [16, 17])
def test_adjoint_and_vjp(n, bits, tol):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    from oracle import lq_oracle as O
    rng = np.random.default_rng([n, bits])
    ops = circuit(n, rng)
    oops = oracle_ops(ops)
    psi = O.apply_ops(O.zero_state(n), n, oops)
    tp = list(range(sum(1 for o in ops if o.params)))
    ref = np.asarray(O.adjoint_jacobian(psi, n, oops, [("N", "PauliY", 2), ("N", "PauliZ", n - 1)], tp)).reshape(2, -1)
    sfx = f"C{bits}"
    sv = getattr(L, "StateVector" + sfx)(n)
    lst = W.to_ops(ops, bits)
    obs = [getattr(L, "NamedObs" + sfx)("PauliY", [2]), getattr(L, "NamedObs" + sfx)("PauliZ", [n - 1])]
    for _ in range(2):
        sv.resetStateVector()
        W.apply_circuit(sv, ops)
        np.testing.assert_allclose(sv.state(), psi, rtol=0, atol=1e-12 if bits == 128 else 1e-5)
        jac = np.asarray(getattr(L.algorithms, "AdjointJacobian" + sfx)()(sv, obs, lst, tp)).reshape(2, -1)
        np.testing.assert_allclose(jac, ref, rtol=0, atol=tol)
        # <Y_2> and its gradient from the vector-Jacobian product: 2 Re <Y psi|d psi>
        dy = O.apply_ops(psi.copy(), n, [O.Op("PauliY", [2], [])]).astype(np.complex128 if bits == 128 else np.complex64)
        vjp = np.asarray(getattr(L.algorithms, "VectorJacobianProduct" + sfx)()(sv, lst, dy, tp))
        np.testing.assert_allclose(2 * vjp.real, ref[0], rtol=0, atol=tol)
        L.jit_wait()


@pytest.mark.parametrize("n", [16])
def test_not_unitary_before_expectations(n):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    from oracle import lq_oracle as O
    rng = np.random.default_rng(n)
    for matrix in (np.array([[0.5, 0.2], [0.1j, 1.5]]), np.diag([0.5, 2.0j])):
        ops = circuit(n, rng, matrix.astype(np.complex128))
        psi = O.apply_ops(O.zero_state(n), n, oracle_ops(ops))
        sv = L.StateVectorC128(n)
        m = L.MeasurementsC128(sv)
        for _ in range(2):
            sv.resetStateVector()
            W.apply_circuit(sv, ops)
            sv.synchronize()
            names = [("PauliZ", "PauliX", "PauliY", "Hadamard")[w % 4] for w in range(n)]
            got = m.expval_named_batch(names, list(range(n)))
            exp = [O.expval_named(psi, n, names[w], [w]) for w in range(n)]
            np.testing.assert_allclose(got, exp, rtol=0, atol=1e-11 * float(np.vdot(psi, psi).real))
            L.jit_wait()
