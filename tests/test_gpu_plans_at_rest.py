"""Plans at rest are lent to one program at a time: threads that run circuits of
one structure with their own angles, and a recording that keeps its plan while
eager runs of the same circuit go on."""
import threading

import numpy as np
import pytest

from helpers import TOL_C128, TOL_C64, ham_to_oracle, oracle_run
from oracle import lq_oracle as O

pytestmark = pytest.mark.gpu

L = pytest.importorskip("lightning_amd.lightning_qubit_ops")
W = pytest.importorskip("lightning_amd.workloads")


@pytest.mark.parametrize("bits,tol", [(128, TOL_C128), (64, TOL_C64)])
def test_threads_of_one_structure(bits, tol):
    n, threads, rounds = 16, 4, 6
    coeffs, words = W.random_pauli_hamiltonian(n, 6, seed=2)
    circuits = [W.hea_rot_cz(n, 3, seed=s) for s in range(threads)]
    states = [oracle_run(n, c) for c in circuits]
    energies = [O.expval_obs(s, n, ham_to_oracle(coeffs, words)) for s in states]
    make, meas = getattr(L, f"StateVectorC{bits}"), getattr(L, f"MeasurementsC{bits}")

    def run(sv, c):
        sv.resetStateVector()
        W.apply_circuit(sv, c)

    sv = make(n)
    run(sv, circuits[0])
    sv.synchronize()
    L.jit_wait()
    run(sv, circuits[0])  # the plan is complete now
    sv.synchronize()
    start, errors = threading.Barrier(threads), []

    def work(k):
        try:
            own = make(n)
            m, ham = meas(own), W.hamiltonian_obs(coeffs, words, bits)
            start.wait()
            for r in range(rounds):
                j = (k + r) % threads  # angles change from round to round
                run(own, circuits[j])
                np.testing.assert_allclose(own.state(), states[j], rtol=0, atol=tol)
                assert abs(m.expval(ham) - energies[j]) < 10 * tol
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[0]


@pytest.mark.parametrize("bits,tol", [(128, TOL_C128), (64, TOL_C64)])
def test_a_recording_keeps_its_plan(bits, tol):
    n = 16
    make = getattr(L, f"StateVectorC{bits}")
    flat = lambda ops: [p for o in ops for p in o.params]  # noqa: E731
    circuits = [W.hea_rot_cz(n, 2, seed=s) for s in range(3)]
    states = [oracle_run(n, c) for c in circuits]
    sv, other = make(n), make(n)
    for _ in range(2):
        other.resetStateVector()
        W.apply_circuit(other, circuits[0])
        other.synchronize()
        L.jit_wait()
    rec = sv.record(W.to_ops(circuits[0], bits))
    for k in range(6):
        # eager runs of the same structure borrow and give back plans meanwhile
        other.resetStateVector()
        W.apply_circuit(other, circuits[(k + 1) % 3])
        rec.replay(flat(circuits[k % 3]))
        np.testing.assert_allclose(other.state(), states[(k + 1) % 3], rtol=0, atol=tol)
        np.testing.assert_allclose(sv.state(), states[k % 3], rtol=0, atol=tol)
