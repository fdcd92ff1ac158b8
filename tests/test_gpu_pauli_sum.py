"""Pauli sums at the edges of the kernel: below one workgroup of amplitudes,
around the change from one to four amplitudes per thread (18 qubits), words
without X or Y, words whose highest flipped bit is a lane, an amplitude of the
thread or a workgroup bit, and repeated words."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def word_masks(n, word):
    """(flipped bits, phase bits, number of Y) of [(name, wire)] on distinct wires."""
    x = z = ny = 0
    for name, w in word:
        b = 1 << (n - 1 - w)
        x |= b if name in ("PauliX", "PauliY") else 0
        z |= b if name in ("PauliZ", "PauliY") else 0
        ny += name == "PauliY"
    return x, z, ny


def apply_sum(psi, n, coeffs, words):
    idx = np.arange(1 << n, dtype=np.uint64)
    out = np.zeros_like(psi, dtype=np.complex128)
    for c, word in zip(coeffs, words):
        x, z, ny = word_masks(n, word)
        par = idx & np.uint64(z)
        for s in (32, 16, 8, 4, 2, 1):
            par = par ^ (par >> np.uint64(s))
        sign = 1.0 - 2.0 * (par & np.uint64(1)).astype(np.float64)
        # P|j> = i^ny (-1)^popcount(j & z)|j ^ x>, so (P psi)_i = (-i)^ny (-1)^popcount(i & z) psi_(i ^ x)
        out += c * (-1j) ** ny * sign * psi[idx ^ np.uint64(x)]
    return out


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 13, 17, 18, 19, 21])
def test_pauli_sum(n, bits):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    rng = np.random.default_rng([n, bits])
    names = ("PauliX", "PauliY", "PauliZ")
    words = [[("Identity", 0)], [("PauliZ", 0)], [("PauliX", n - 1)], [("PauliY", 0)]]
    words += [[(names[k % 3], n - 1 - b)] for k, b in enumerate((7, 8, 9, 10)) if b < n]
    while len(words) < 40:  # more than the dots of one pass: the sum runs in its own kernel
        letters = rng.choice(4, size=n, p=[0.4, 0.2, 0.2, 0.2])
        words.append([(names[c - 1], w) for w, c in enumerate(letters) if c] or [("PauliY", n - 1)])
    words += words[5:7]
    coeffs = [float(c) for c in rng.standard_normal(len(words))]
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex128 if bits == 128 else np.complex64)
    sv = (L.StateVectorC128 if bits == 128 else L.StateVectorC64)(n)
    sv.updateData(psi)
    m = (L.MeasurementsC128 if bits == 128 else L.MeasurementsC64)(sv)
    ham = W.hamiltonian_obs(coeffs, words, bits)
    h = apply_sum(psi.astype(np.complex128), n, coeffs, words)
    e = np.vdot(psi.astype(np.complex128), h).real
    total = sum(abs(c) for c in coeffs)
    # FP64 arithmetic in both precisions: each word's mean is off by at most some 2^8 units of its size
    assert abs(m.expval(ham) - e) < 2.0 ** 8 * 2.3e-16 * total
    # H psi is rounded to the state's precision before its norm is taken
    eps = 2.0 ** 8 * 2.3e-16 if bits == 128 else 4 * 6e-8
    assert abs(m.var(ham) - (np.vdot(h, h).real - e * e)) < 2 * eps * total ** 2

