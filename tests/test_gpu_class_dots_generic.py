"""X, Y and Z dots in the interpreting register kernel (11 to 15 qubits are
never specialised): the adjoint's imaginary parts and the expectations' real
parts, with targets on register, thread and outside bits and with controls,
which take the general form.

Tolerance: the oracle's double-precision sums and some 150 unitary ops, each
off by a few 2^-53 (complex64: 2^-24) in amplitudes of norm 1, and an
observable of norm 1: 1e-11 and 5e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,tol", [(128, 1e-11), (64, 5e-4)])
@pytest.mark.parametrize("n", [11, 12, 13, 15])
def test_class_dots(n, bits, tol):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    from oracle import lq_oracle as O
    rng = np.random.default_rng([7, n, bits])
    ops = []
    for layer in range(2):
        for w in range(n):
            ops += [W.CircuitOp(g, [w], [float(rng.uniform(-3, 3))]) for g in ("RX", "RY", "RZ")]
        for w in range(n - 1):
            ops.append(W.CircuitOp("CNOT" if layer else "CZ", [w, w + 1]))
        ops += [W.CircuitOp("CRX", [0, n - 1], [0.3]), W.CircuitOp("CRZ", [n - 1, 1], [0.7])]
    oops = [O.Op(o.name, o.wires, o.params, o.inverse, o.matrix, o.ctrls, o.cvals) for o in ops]
    psi = O.apply_ops(O.zero_state(n), n, oops)
    tp = list(range(sum(1 for o in ops if o.params)))
    want = np.asarray(O.adjoint_jacobian(psi, n, oops, [("N", "PauliY", 1)], tp)).reshape(-1)
    sfx = f"C{bits}"
    sv = getattr(L, "StateVector" + sfx)(n)
    W.apply_circuit(sv, ops)
    jac = getattr(L.algorithms, "AdjointJacobian" + sfx)()(
        sv, [getattr(L, "NamedObs" + sfx)("PauliY", [1])], W.to_ops(ops, bits), tp)
    np.testing.assert_allclose(np.asarray(jac).reshape(-1), want, rtol=0, atol=tol)
    names = [("PauliX", "PauliY", "PauliZ")[w % 3] for w in range(n)]
    got = getattr(L, "Measurements" + sfx)(sv).expval_named_batch(names, list(range(n)))
    np.testing.assert_allclose(got, [O.expval_named(psi, n, names[w], [w]) for w in range(n)], rtol=0, atol=tol)
