"""Dense operators on three to six wires, which run in passes of their own
(tiles of eleven bits): targets on the lowest and highest index bits and
between, in any wire order, with controls inside and outside the tile, at the
smallest sizes that take the pass and those just below it, inverse, between
other gates, and on the two states of an adjoint sweep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def haar(dim, rng):
    z = rng.standard_normal((dim, dim)) + 1j * rng.standard_normal((dim, dim))
    q, r = np.linalg.qr(z)
    return q * (np.diag(r) / np.abs(np.diag(r)))


def apply(psi, n, mat, wires, ctrls=(), values=()):
    """mat on `wires` where the controls hold their values (complex128)."""
    rest = [w for w in range(n) if w not in wires and w not in ctrls]
    order = list(ctrls) + list(wires) + rest
    t = psi.reshape([2] * n).transpose(order).copy().reshape((2,) * len(ctrls) + (1 << len(wires), -1))
    sel = tuple(int(v) for v in values)
    t[sel] = mat @ t[sel]
    back = np.argsort(order)
    return t.reshape([2] * n).transpose(back).reshape(-1)


def placements(n, k):
    yield list(range(n - k, n)), [], []            # lowest bits: lanes of the load are targets
    yield list(range(n - 1, n - 1 - k, -1)), [], []  # the same, reversed
    yield list(range(k)), [], []                   # highest bits
    yield [0, n - 1] + list(range(3, 1 + k)), [], []
    yield list(range(1, k + 1)), [n - 1], [0]      # a control on the lowest bit: inside the tile
    yield list(range(n - k, n)), [0], [1]          # outside
    yield list(range(2, k + 2)), [n - 2, 0, n - 4], [1, 0, 1]


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("k", [3, 4, 5, 6])
@pytest.mark.parametrize("n", [10, 11, 12, 13, 16])
def test_dense_operator(n, k, bits):
    from lightning_amd import lightning_qubit_ops as L
    cdt = np.complex128 if bits == 128 else np.complex64
    rng = np.random.default_rng([n, k, bits])
    # rounding of one operator: sums of 2^(k+1) <= 2^7 products in the state's precision, of
    # amplitudes of total norm one, plus the rounding of the inputs to that precision
    tol = 2.0 ** 8 * (1.2e-16 if bits == 128 else 6e-8) * 8 * 2.0 ** (-n / 2)
    for i, (wires, ctrls, values) in enumerate(placements(n, k)):
        if set(wires) & set(ctrls) or max(wires) >= n:
            continue
        psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
        psi = (psi / np.linalg.norm(psi)).astype(cdt)
        mat = haar(1 << k, rng).astype(cdt)
        sv = (L.StateVectorC128 if bits == 128 else L.StateVectorC64)(n)
        sv.updateData(psi)
        inverse = i % 2 == 1
        if ctrls:
            sv.applyControlledMatrix(mat, ctrls, [bool(v) for v in values], wires, inverse)
        else:
            sv.applyMatrix(mat, wires, inverse)
        m = mat.astype(np.complex128)
        exp = apply(psi.astype(np.complex128), n, m.conj().T if inverse else m, wires, ctrls, values)
        np.testing.assert_allclose(sv.state(), exp, rtol=0, atol=tol, err_msg=f"{wires} {ctrls} {values} {inverse}")


@pytest.mark.parametrize("n", [12, 17])
def test_between_gates_and_in_a_gradient(n):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    from oracle import lq_oracle as O
    rng = np.random.default_rng(n)
    ops = W.strongly_entangling(n, 1, seed=n)
    for k in (3, 5, 4):
        wires = [int(w) for w in rng.choice(n, size=k, replace=False)]
        ops.insert(len(ops) // 2, W.CircuitOp("QubitUnitary", wires, [0.0], matrix=haar(1 << k, rng)))
    ops += W.strongly_entangling(n, 1, seed=n + 1)
    sv = L.StateVectorC128(n)
    W.apply_circuit(sv, ops)
    oops = [O.Op(o.name, o.wires, o.params, o.inverse, o.matrix) for o in ops]
    psi = O.apply_ops(O.zero_state(n), n, oops)
    np.testing.assert_allclose(sv.state(), psi, rtol=0, atol=1e-12)
    par = [i for i, o in enumerate([o for o in ops if o.params]) if o.matrix is None]
    obs = [L.NamedObsC128("PauliX", [3]), L.NamedObsC128("PauliZ", [n - 1])]
    jac = np.asarray(L.AdjointJacobianC128()(sv, obs, W.to_ops(ops), par)).reshape(2, -1)
    ref = np.asarray(O.adjoint_jacobian(psi, n, oops, [("N", "PauliX", 3), ("N", "PauliZ", n - 1)], par))
    np.testing.assert_allclose(jac, ref, rtol=0, atol=1e-10)
