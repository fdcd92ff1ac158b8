"""Marginals with more items than workgroups: nearly all high bits measured, in
order and not, with and without low bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(21, list(range(13))), (22, list(range(16))), (22, [3, 21, 9, 0, 12, 11, 2, 16, 5, 13, 7, 10, 1, 4, 6, 8]),
         (22, list(range(21, -1, -1))), (21, list(range(21)))]


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("n,wires", CASES)
def test_probs_of_many_items(n, wires, bits):
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
    # sums of at most 2^9 positive FP64 terms; complex64 results are rounded to float32
    np.testing.assert_allclose(got, exp, rtol=2.0 ** 9 * 2.3e-16 if bits == 128 else 1.2e-7, atol=0)
