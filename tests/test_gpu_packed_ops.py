"""The packed request kernel in each of its workgroup sizes (256 threads up to
9 qubits, 512 at 10, 1024 from 11 and for states in global memory) and with
every kind of op it runs, against the oracle.

Tolerance: some 40 unitary ops and 40-odd terms in double precision, a few
units of 2^-53 each: 1e-12 (complex64: 2^-24, 5e-5)."""
import numpy as np
import pytest

from helpers import ham_to_oracle, oracle_run, to_oracle_ops
from oracle import lq_oracle as O

pytestmark = pytest.mark.gpu

S = pytest.importorskip("lightning_amd.serving")
W = pytest.importorskip("lightning_amd.workloads")


def request(n, bits):
    rng = np.random.default_rng([41, n])
    ang = iter(rng.uniform(-3.0, 3.0, size=1000))
    ops = [W.CircuitOp("RY", [w], [next(ang)]) for w in range(n)] + [W.CircuitOp("Hadamard", [0])]
    for _ in range(2):
        if n > 1:
            for name in ("IsingXX", "IsingZZ", "CRY", "ControlledPhaseShift", "IsingXY", "SingleExcitation"):
                a, b = (int(x) for x in rng.permutation(n)[:2])
                ops.append(W.CircuitOp(name, [a, b], [next(ang)]))
            ops.append(W.CircuitOp("SWAP", [0, n - 1]))
        ops += [W.CircuitOp("RX", [n - 1], [next(ang)]), W.CircuitOp("PhaseShift", [0], [next(ang)])]
    H = O.random_pauli_hamiltonian(n, 7, seed=n, probs_ixyz=(0.4, 0.2, 0.2, 0.2))
    return S.Request(n, 2, ops, list(H[1]), [list(t[1]) for t in H[2]], bits)


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("n", [1, 2, 7, 9, 10, 11, 12, 13, 14])
def test_packed_ops(n, bits):
    req = request(n, bits)
    srv = S.Server(bits=bits, batched=True, small_max_qubits=14)
    energy, grad = srv.run(req)[:2]
    packed = srv.stats()["packed"]
    srv.close()
    assert packed == 1
    st = oracle_run(n, req.ops)
    H = ham_to_oracle(req.coeffs, req.words)
    want = O.adjoint_jacobian(st, n, to_oracle_ops(req.ops), [H], list(range(req.num_params)))[0]
    tol = 1e-12 if bits == 128 else 5e-5
    scale = sum(abs(c) for c in req.coeffs)
    assert abs(energy - O.expval_obs(st, n, H)) < tol * scale
    np.testing.assert_allclose(grad, want, rtol=0, atol=tol * scale)
