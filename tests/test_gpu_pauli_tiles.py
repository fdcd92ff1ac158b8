"""Sums of many Pauli words on 24 qubits (the kernel that takes a group of words
from one tile in LDS) and around its limits: 23 qubits, complex64 and few words
take the other kernel. On the product state of RY(t_q) RZ(p_q), a word's mean
is the product of sin t cos p (X), sin t sin p (Y) and cos t (Z).

Tolerance: words times 2^5 units of the precision of the states (each gradient
is one sum over amplitudes of norm 1, formed in double precision): 60 * 2^5 *
1.1e-16 and, for complex64 states, 6e-8 in place of 1.1e-16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ("PauliX", "PauliY", "PauliZ")


@pytest.mark.parametrize("n,terms,bits", [(24, 32, 128), (24, 60, 128), (24, 31, 128), (23, 40, 128), (24, 40, 64)])
def test_gradient_of_a_sum(n, terms, bits):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    rng = np.random.default_rng([n, terms, bits])
    t, p = rng.uniform(0.4, 2.7, n), rng.uniform(-3, 3, n)
    coeffs = rng.standard_normal(terms)
    words = []
    for k in range(terms):
        r = rng.integers(0, 8 if k % 3 else 24, size=n)
        words.append([(NAMES[r[w]], w) for w in range(n) if r[w] < 3] or [("PauliY", k % n)])
    words[1] = words[0]  # a repeated word, and one that differs in its low bits
    words[2] = [f for f in words[0] if f[1] != n - 1] + [("PauliX", n - 1)]
    f = {"PauliX": np.sin(t) * np.cos(p), "PauliY": np.sin(t) * np.sin(p), "PauliZ": np.cos(t)}
    dt = {"PauliX": np.cos(t) * np.cos(p), "PauliY": np.cos(t) * np.sin(p), "PauliZ": -np.sin(t)}
    dp = {"PauliX": -np.sin(t) * np.sin(p), "PauliY": np.sin(t) * np.cos(p), "PauliZ": np.zeros(n)}
    want = np.zeros((n, 2))
    for c, word in zip(coeffs, words):
        for name, w in word:
            rest = np.prod([f[o][v] for o, v in word if v != w])
            want[w] += c * rest * np.array([dt[name][w], dp[name][w]])
    ops = [W.CircuitOp(g, [w], [float(a[w])]) for w in range(n) for g, a in (("RY", t), ("RZ", p))]
    sfx = f"C{bits}"
    sv = getattr(L, "StateVector" + sfx)(n)
    W.apply_circuit(sv, ops)
    jac = getattr(L.algorithms, "AdjointJacobian" + sfx)()(
        sv, [W.hamiltonian_obs([float(c) for c in coeffs], words, bits)], W.to_ops(ops, bits), list(range(2 * n)))
    tol = terms * 32 * (1.1e-16 if bits == 128 else 6e-8)
    np.testing.assert_allclose(np.asarray(jac).reshape(n, 2), want, rtol=0, atol=tol)
