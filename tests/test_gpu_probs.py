"""Marginal probabilities at the edges of the kernel's split of the index (low
eight bits per thread, measured high bits per workgroup, unmeasured ones
summed per thread or split over rows): sizes below and above eight qubits, few
and many wires, wires on either side of the edge, in any order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    (1, [0]), (3, [2, 0]), (6, [5, 1, 3]), (7, [0, 6]), (7, [3]), (8, [0]), (8, [7, 0, 1]), (9, [0]), (9, [8, 1]),
    (12, list(range(12))), (12, list(range(11, -1, -1))), (13, [12]), (13, [5, 6, 4]), (16, [15, 14, 13, 12, 11, 10, 9, 8]),
    (16, [0, 1, 2, 3, 4, 5, 6, 7]), (18, [3, 17, 9, 0, 11, 10, 2, 16, 5, 12, 7]), (20, [19, 0]),
    (20, [1, 18, 3, 16, 5, 14, 7, 12, 9, 10, 11, 0, 13]), (20, list(range(0, 10))), (21, [4]), (21, list(range(2, 19))),
]


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("n,wires", CASES)
def test_probs_match_marginals(n, wires, bits):
    from lightning_amd import lightning_qubit_ops as L
    rng = np.random.default_rng([n, len(wires), bits])
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex128 if bits == 128 else np.complex64)
    sv = (L.StateVectorC128 if bits == 128 else L.StateVectorC64)(n)
    sv.updateData(psi)
    got = (L.MeasurementsC128 if bits == 128 else L.MeasurementsC64)(sv).probs(wires)
    p = np.square(psi.real, dtype=np.float64) + np.square(psi.imag, dtype=np.float64)
    rest = [w for w in range(n) if w not in wires]
    exp = p.reshape([2] * n).transpose(wires + rest).reshape(1 << len(wires), -1).sum(axis=1)
    # sums of at most 2^21 positive FP64 terms of total 1, per thread in four chains of at most
    # 2^9 terms, then trees: below 2^10 units in the last place; complex64 results are rounded to float32
    tol = 2.0 ** 10 * 2.3e-16
    np.testing.assert_allclose(got, exp, rtol=tol if bits == 128 else 1.2e-7, atol=0)
    again = (L.MeasurementsC128 if bits == 128 else L.MeasurementsC64)(sv).probs(wires)
    np.testing.assert_array_equal(got, again)
