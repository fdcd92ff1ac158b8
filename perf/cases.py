"""Measured workloads of the state-vector engine, through its public entry points.

Four kinds of work that programs on this engine do, from calls of a few
microseconds of GPU work to states that fill a good part of the card:

* ``circuit``: reset, a parametrised circuit, and its results (expectation
  values of every wire, the probabilities of some wires, or the state).
* ``gradient``: the circuit's energies and their adjoint Jacobian, as one step
  of a variational optimisation; ``training`` is the same through the torch
  function with its backward pass.
* ``measure`` / ``matrix``: a prepared state that is measured (probabilities,
  Pauli sums, a Hermitian matrix, a variance, samples), and dense matrices of
  one to six wires, some controlled, that are applied to it.
* ``serve``: a burst of small energy + gradient requests of the request server.

Sizes are those of the repository's benchmark, examples and tests (10-qubit
smoke circuit, 20-qubit RX/RY/RZ+CNOT, 24-qubit 432-parameter gradient, 30-qubit
hardware-efficient ansatz, serving requests) with odd sizes between them.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pennylane-lightning_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

# Circuits of the repository's workloads: (name, most qubits drawn).
ANSAETZE = ("rxyz_cnot", "hea", "strong", "qft")


def listed():
    return [
        # the first circuit anyone runs: 10 qubits, three layers, <Z> of every
        # wire; launches and host work count
        {"name": "circuit_10", "kind": "circuit", "ansatz": "rxyz_cnot", "n": 10, "layers": 3, "bits": 128,
         "result": "expval"},
        # 20 qubits, ten layers of RX RY RZ + CNOT, <Z> and probabilities of ten wires
        {"name": "circuit_20", "kind": "circuit", "ansatz": "rxyz_cnot", "n": 20, "layers": 10, "bits": 128,
         "result": "probs"},
        # QFT, Haar 4x4 brickwork and multi-controlled X in single precision
        {"name": "qft_27_c64", "kind": "circuit", "ansatz": "qft", "n": 27, "layers": 4, "bits": 64,
         "result": "state"},
        # the headline circuit: 30 qubits, 1180 gates, 16 GiB of amplitudes
        {"name": "hea_30", "kind": "circuit", "ansatz": "hea", "n": 30, "layers": 20, "bits": 128,
         "result": "state"},
        # a variational step on a few qubits: energy and gradient of a 50-term Hamiltonian
        {"name": "gradient_13", "kind": "gradient", "ansatz": "hea", "n": 13, "layers": 6, "bits": 128,
         "terms": 50, "observables": 1},
        # the 24-qubit, 432-parameter, 200-term energy and gradient
        {"name": "gradient_24", "kind": "gradient", "ansatz": "strong", "n": 24, "layers": 6, "bits": 128,
         "terms": 200, "observables": 1},
        # the Jacobian of three observables in single precision, an odd size
        {"name": "gradient_21_c64", "kind": "gradient", "ansatz": "hea", "n": 21, "layers": 7, "bits": 64,
         "terms": 1, "observables": 3},
        # one step of a torch training loop: forward and backward pass
        {"name": "training_17", "kind": "training", "ansatz": "strong", "n": 17, "layers": 3, "bits": 128,
         "observables": 4},
        # measurements of a small state, samples among them
        {"name": "measure_15", "kind": "measure", "n": 15, "bits": 128, "wires": 9, "terms": 30, "shots": 1000},
        # measurements of a large state
        {"name": "measure_26", "kind": "measure", "n": 26, "bits": 128, "wires": 14, "terms": 40, "shots": 0},
        # dense operators on one to six wires, plain, inverse and controlled
        {"name": "matrix_23", "kind": "matrix", "n": 23, "bits": 128, "widest": 6},
        # a burst of small requests: the request server's packed path
        {"name": "serve_64", "kind": "serve", "count": 64, "n_min": 10, "n_max": 15, "bits": 128},
    ]


def draw(rng):
    kind = rng.choice(["circuit", "circuit", "gradient", "gradient", "training", "measure", "matrix", "serve"])
    bits = rng.choice([128, 128, 64])
    if kind == "circuit":
        ansatz = rng.choice(ANSAETZE)
        n = rng.randint(4, 28)
        return {"kind": kind, "ansatz": ansatz, "n": n, "layers": rng.randint(1, 10 if n <= 24 else 5), "bits": bits,
                "result": rng.choice(["expval", "probs", "state"])}
    if kind == "gradient":
        n = rng.randint(4, 24)
        return {"kind": kind, "ansatz": rng.choice(["rxyz_cnot", "hea", "strong"]), "n": n,
                "layers": rng.randint(1, 6), "bits": bits, "terms": round(math.exp(rng.uniform(0, math.log(200)))),
                "observables": rng.choice([1, 1, 2, 3])}
    if kind == "training":
        return {"kind": kind, "ansatz": rng.choice(["rxyz_cnot", "hea", "strong"]), "n": rng.randint(4, 22),
                "layers": rng.randint(1, 4), "bits": bits, "observables": rng.randint(1, 5)}
    if kind == "measure":
        n = rng.randint(6, 26)
        return {"kind": kind, "n": n, "bits": bits, "wires": rng.randint(1, min(n, 16)),
                "terms": round(math.exp(rng.uniform(0, math.log(100)))),
                "shots": rng.choice([0, 100, 1000]) if bits == 128 and n <= 20 else 0}
    if kind == "matrix":
        return {"kind": kind, "n": rng.randint(8, 25), "bits": bits, "widest": rng.randint(2, 6)}
    n_min = rng.randint(4, 12)
    return {"kind": kind, "count": round(math.exp(rng.uniform(math.log(4), math.log(64)))), "n_min": n_min,
            "n_max": rng.randint(n_min, 15), "bits": bits}


# ---------------------------------------------------------------------------
# Inputs (numbers only; shared with the 64-bit results below)
# ---------------------------------------------------------------------------
def _circuit_ops(case, seed, adjoint_form):
    from lightning_amd import workloads as W
    n, layers = case["n"], case["layers"]
    if case["ansatz"] == "rxyz_cnot":
        return W.layers_rxyz_cnot(n, layers, seed)
    if case["ansatz"] == "strong":
        return W.strongly_entangling(n, layers, seed)
    if case["ansatz"] == "hea":
        return (W.hea_rot_cz_adjoint_form if adjoint_form else W.hea_rot_cz)(n, layers, seed)
    # where the multi-controlled gates sit is the circuit's, the matrices are the seed's
    ops = W.qft_brickwork_mcx(n, layers, 1, 5)
    rng = np.random.default_rng(seed)
    for op in ops:
        if op.matrix is not None:
            op.matrix = W.haar_unitary(4, rng)
        elif op.name == "ControlledPhaseShift":
            op.params = [op.params[0] * rng.uniform(0.5, 1.0)]
    return ops


def _pauli_sums(case, seed):
    """One (coefficients, words) for each observable; a single word has the coefficient 1, and no word is the identity."""
    from lightning_amd import workloads as W
    out = []
    for k in range(case.get("observables", 1)):
        c, w = W.random_pauli_hamiltonian(case["n"], case.get("terms", 1), seed + 1000 * (k + 1))
        w = [[("PauliZ", 0)] if word == [("Identity", 0)] else word for word in w]
        out.append((c if len(c) > 1 else [1.0], w))
    return out


def _random_state(n, seed, device):
    """Normalised amplitudes with the magnitudes of a random circuit's, complex128."""
    g = torch.Generator(device=device).manual_seed(seed)
    a = torch.randn((1 << n, 2), generator=g, dtype=torch.float64, device=device)
    return torch.view_as_complex(a / torch.linalg.vector_norm(a))


def _state_dtype(case):
    return torch.complex128 if case["bits"] == 128 else torch.complex64


def _hermitian(dim, rng):
    m = rng.standard_normal((dim, dim)) + 1j * rng.standard_normal((dim, dim))
    return (m + m.conj().T) / (2 * math.sqrt(dim))


def _measure_inputs(case, seed):
    n = case["n"]
    # which wires are read is the program's, the values are the seed's
    place = np.random.default_rng([7, n, case["wires"]])
    wires = [int(w) for w in place.choice(n, size=case["wires"], replace=False)]
    pair = [int(w) for w in place.choice(n, size=2, replace=False)]
    rng = np.random.default_rng(seed)
    return wires, pair, _hermitian(4, rng), _pauli_sums(case, seed)[0]


def _matrix_ops(case, seed):
    """(matrix, wires, controls, values, inverse) in the order of application."""
    from lightning_amd import workloads as W
    n = case["n"]
    place = np.random.default_rng([11, n, case["widest"]])
    rng = np.random.default_rng(seed)
    out = []
    for k in range(1, case["widest"] + 1):
        for nc in (0, 1 if k % 2 else 2):
            at = [int(w) for w in place.choice(n, size=min(k + nc, n), replace=False)]
            out.append((W.haar_unitary(1 << k, rng), at[:k], at[k:], [bool(place.integers(2)) for _ in at[k:]],
                        bool(k % 3 == 0)))
    return out


def _requests(case, seed):
    from lightning_amd import serving as S
    # the sizes and depths of the burst are the case's, angles and Hamiltonians the seed's
    place = np.random.default_rng([13, case["count"], case["n_min"], case["n_max"]])
    out = []
    for i in range(case["count"]):
        n, depth = int(place.integers(case["n_min"], case["n_max"] + 1)), int(place.integers(4, 13))
        rng = np.random.default_rng([seed, i])
        ops = S.hea_adjoint_ops(n, depth, rng)
        coeffs, words = S.random_pauli_hamiltonian(n, 50, seed=int(rng.integers(1 << 31)))
        out.append(S.Request(n, depth, ops, coeffs, words, case["bits"]))
    return out


# ---------------------------------------------------------------------------
# The framework's side
# ---------------------------------------------------------------------------
_SERVERS = {}


def _server(bits):
    """A program keeps one request server running for all its bursts."""
    from lightning_amd import serving as S
    if bits not in _SERVERS:
        _SERVERS[bits] = S.Server(bits=bits)
    return _SERVERS[bits]


def prepare(case, seed):
    from lightning_amd import lightning_qubit_ops as L
    from lightning_amd import workloads as W
    kind, bits = case["kind"], case["bits"]
    s = {"case": case}
    if kind == "serve":
        s["requests"] = _requests(case, seed)
        for r in s["requests"]:
            r.handles()
        s["arrivals"] = np.zeros(len(s["requests"]))
        s["server"] = _server(bits)
        return s
    n = case["n"]
    if kind == "training":
        ops = _circuit_ops(case, seed, True)
        s["ops"] = ops
        s["params"] = torch.tensor([v for op in ops for v in op.params], dtype=torch.float64)
        s["observables"] = [("N", ("PauliX", "PauliY", "PauliZ")[k % 3], (5 * k) % n)
                            for k in range(case["observables"])]
    else:
        s["sv"] = (L.StateVectorC128 if bits == 128 else L.StateVectorC64)(n)
        s["m"] = (L.MeasurementsC128 if bits == 128 else L.MeasurementsC64)(s["sv"])
    if kind == "circuit":
        s["ops"] = _circuit_ops(case, seed, False)
    elif kind == "gradient":
        s["ops"] = _circuit_ops(case, seed, True)
        s["list"] = W.to_ops(s["ops"], bits)
        s["obs"] = [W.hamiltonian_obs(c, w, bits) for c, w in _pauli_sums(case, seed)]
        s["trainable"] = list(range(sum(1 for o in s["ops"] if o.params)))
        s["adjoint"] = (L.algorithms.AdjointJacobianC128 if bits == 128 else L.algorithms.AdjointJacobianC64)()
    elif kind in ("measure", "matrix"):
        s["psi"] = _random_state(n, seed, "cuda").to(_state_dtype(case))
        s["sv"].updateData(s["psi"])
        if kind == "measure":
            wires, pair, herm, (coeffs, words) = _measure_inputs(case, seed)
            s.update(wires=wires, pair=pair, herm=herm, ham=W.hamiltonian_obs(coeffs, words, bits))
            s["word"] = W.hamiltonian_obs([1.0], words[:1], bits)
            s["m"].set_random_seed(seed)
        else:
            s["ops"] = _matrix_ops(case, seed)
    if kind in ("circuit", "gradient", "training") and n >= 16:
        # a program that repeats a circuit has its kernels compiled after the
        # first passes; the second one may ask for more (several observables)
        for _ in range(2):
            run(s)
            L.jit_wait()
    return s


def run(s):
    from lightning_amd import workloads as W
    case = s["case"]
    kind = case["kind"]
    if kind == "serve":
        r = s["server"].replay(s["requests"], s["arrivals"])
        return {"energies": r["energies"], "gradients": np.concatenate(r["grads"])}
    if kind == "training":
        from lightning_amd.torch_interface import circuit_expvals
        p = s["params"].clone().requires_grad_(True)
        ev = circuit_expvals(p, case["n"], s["ops"], s["observables"], case["bits"])
        (ev * ev).sum().backward()
        return {"expvals": ev.detach(), "gradient": p.grad}
    sv, m, n = s["sv"], s["m"], case["n"]
    if kind == "circuit":
        sv.resetStateVector()
        W.apply_circuit(sv, s["ops"])
        if case["result"] == "state":
            return {"state": sv.to_torch()}
        out = {"z": m.expval_named_batch(["PauliZ"] * n, list(range(n)))}
        if case["result"] == "probs":
            out["probs"] = m.probs(list(range(min(n, 10))))
        return out
    if kind == "gradient":
        sv.resetStateVector()
        W.apply_circuit(sv, s["ops"])
        jac, energy = s["adjoint"](sv, s["obs"], s["list"], s["trainable"], return_expvals=True)
        return {"jacobian": jac, "energy": energy}
    if kind == "matrix":
        sv.updateData(s["psi"])
        for mat, wires, ctrls, values, inverse in s["ops"]:
            if ctrls:
                sv.applyControlledMatrix(mat, ctrls, values, wires, inverse)
            else:
                sv.applyMatrix(mat, wires, inverse)
        return {"state": sv.to_torch()}
    out = {"probs": m.probs(s["wires"]), "energy": m.expval(s["ham"]), "x": m.expval("PauliX", [s["pair"][0]]),
           "hermitian": m.expval(s["herm"], s["pair"]), "variance": m.var(s["word"])}
    if case["shots"]:
        out["samples"] = m.generate_samples(s["wires"], case["shots"])
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
# floating-point operations per amplitude of a gate applied once
_GATE_FLOPS = {"RX": 6, "RY": 6, "RZ": 6, "Rot": 14, "Hadamard": 4, "ControlledPhaseShift": 1.5}


def _ops_flops(ops, n):
    total = 0.0
    for op in ops:
        if op.matrix is not None:
            total += 8.0 * (1 << len(op.wires)) - 2
        else:
            total += _GATE_FLOPS.get(op.name, 0)
    return total * 2.0 ** n


def work(case):
    kind = case["kind"]
    size = case["bits"] // 8
    if kind == "serve":
        # forward, inverse gates on two states, one dot for each angle, the Hamiltonian once
        flops, values = 0.0, 0
        for r in _requests(case, 0):
            flops += 3 * _ops_flops(r.ops, r.n) + (4.0 * r.num_params + 400.0) * 2.0 ** r.n
            values += r.num_params
        return {"bytes": 16.0 * values, "flops": flops}
    n = case["n"]
    amps = 2.0 ** n
    if kind == "circuit":
        flops = _ops_flops(_circuit_ops(case, 0, False), n)
        return {"bytes": size * amps, "flops": flops + (4.0 * amps if case["result"] != "state" else 0.0)}
    if kind in ("gradient", "training"):
        ops = _circuit_ops(case, 0, True)
        m = case["observables"] if kind == "gradient" else 1
        trainable = sum(1 for o in ops if o.params)
        # lambda and one state for each observable are written once and read once
        return {"bytes": 2.0 * size * (1 + m) * amps,
                "flops": (2 + m) * _ops_flops(ops, n) + (4.0 * trainable + 8.0 * case.get("terms", 1)) * m * amps}
    if kind == "matrix":
        flops = sum((8.0 * m.shape[0] - 2) / (1 << len(c)) for m, _, c, _, _ in _matrix_ops(case, 0))
        return {"bytes": 2.0 * size * amps, "flops": flops * amps}
    # five results, each of which reads the state
    return {"bytes": 5.0 * size * amps + 8.0 * (1 << case["wires"]), "flops": (8.0 * case["terms"] + 60.0) * amps}


# ---------------------------------------------------------------------------
# The same results in plain torch, 64 bits
# ---------------------------------------------------------------------------
_X = np.array([[0, 1], [1, 0]], complex)
_PAULI = {"PauliX": _X, "PauliY": np.array([[0, -1j], [1j, 0]]), "PauliZ": np.diag([1.0 + 0j, -1.0])}


def _matrix_of(op):
    """The matrix of a gate on its own wires (controls of CNOT and the like included)."""
    if op.matrix is not None:
        return np.asarray(op.matrix)
    t = op.params[0] if op.params else 0.0
    c, s = math.cos(t / 2), math.sin(t / 2)
    if op.name == "RX":
        return np.array([[c, -1j * s], [-1j * s, c]])
    if op.name == "RY":
        return np.array([[c, -s], [s, c]], complex)
    if op.name == "RZ":
        return np.diag([c - 1j * s, c + 1j * s])
    if op.name == "Rot":
        phi, theta, omega = op.params
        z = lambda v: np.diag([np.exp(-0.5j * v), np.exp(0.5j * v)])  # noqa: E731
        c, s = math.cos(theta / 2), math.sin(theta / 2)
        return z(omega) @ np.array([[c, -s], [s, c]]) @ z(phi)
    if op.name == "Hadamard":
        return np.array([[1, 1], [1, -1]], complex) / math.sqrt(2)
    if op.name == "CNOT":
        return np.eye(4, dtype=complex)[[0, 1, 3, 2]]
    if op.name == "CZ":
        return np.diag([1.0 + 0j, 1, 1, -1])
    if op.name == "SWAP":
        return np.eye(4, dtype=complex)[[0, 2, 1, 3]]
    if op.name == "ControlledPhaseShift":
        return np.diag([1.0 + 0j, 1, 1, np.exp(1j * t)])
    return _PAULI[op.name]


def _blocks(psi, n, wires):
    """psi as a view with one dimension of two for each of `wires` (at 1, 3, 5, ... in wire order)."""
    shape, last = [], -1
    for w in sorted(wires):
        shape += [1 << (w - last - 1), 2]
        last = w
    return psi.view(shape + [1 << (n - 1 - last)])


def _apply(psi, n, mat, wires, ctrls=(), values=()):
    """mat on `wires` of psi where the controls hold their values, in place."""
    order = sorted(list(wires) + list(ctrls))
    v = _blocks(psi, n, order)
    at = {w: 1 + 2 * i for i, w in enumerate(order)}
    pick = [slice(None)] * v.dim()
    for w, b in zip(ctrls, values):
        pick[at[w]] = slice(int(b), int(b) + 1)
    v = v[tuple(pick)]
    k = len(wires)
    parts = []
    for i in range(1 << k):
        sel = [slice(None)] * v.dim()
        for j, w in enumerate(wires):
            b = (i >> (k - 1 - j)) & 1
            sel[at[w]] = slice(b, b + 1)
        parts.append(v[tuple(sel)])
    mat = np.asarray(mat)
    if np.count_nonzero(mat - np.diag(np.diag(mat))) == 0:
        for i, p in enumerate(parts):
            if mat[i, i] != 1:
                p *= complex(mat[i, i])
        return psi
    if k <= 2:
        old = [p.clone() for p in parts]
        for r, p in enumerate(parts):
            terms = [(complex(mat[r, c]), old[c]) for c in range(1 << k) if mat[r, c] != 0]
            new = terms[0][1] * terms[0][0]
            for f, x in terms[1:]:
                new.add_(x, alpha=f)
            p.copy_(new)
        return psi
    old = torch.stack([p.reshape(-1) for p in parts])
    new = torch.from_numpy(np.ascontiguousarray(mat, dtype=np.complex128)).to(psi.device) @ old
    for r, p in enumerate(parts):
        p.copy_(new[r].view(p.shape))
    return psi


def _apply_op(psi, n, op, dagger=False):
    mat = _matrix_of(op)
    if dagger != bool(op.inverse):
        mat = mat.conj().T
    return _apply(psi, n, mat, op.wires, op.ctrls, op.cvals or [True] * len(op.ctrls))


def _apply_sum(psi, n, coeffs, words):
    """sum_t c_t P_t psi for Pauli words."""
    out = torch.zeros_like(psi)
    for c, word in zip(coeffs, words):
        v = psi.clone()
        for name, w in word:
            if name != "Identity":
                _apply(v, n, _PAULI[name], [w])
        out.add_(v, alpha=c)
    return out


def _run_exact(ops, n, device):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=device)
    psi[0] = 1
    for op in ops:
        _apply_op(psi, n, op)
    return psi


def _marginal(psi, n, wires):
    """Probabilities of `wires`, the first the most significant bit."""
    p = psi.real.square() + psi.imag.square()
    v = _blocks(p, n, wires)
    v = v.sum(dim=[d for d in range(v.dim()) if d % 2 == 0])
    rank = {w: i for i, w in enumerate(sorted(wires))}
    return v.permute([rank[w] for w in wires]).reshape(-1).cpu().numpy()


def _gradient(ops, n, psi, sums):
    """Energies and their derivatives by each RX, RY, RZ angle: dE/dt = Im <H psi|G psi>."""
    energy, jac = [], []
    for coeffs, words in sums:
        lam = psi.clone()
        mu = _apply_sum(lam, n, coeffs, words)
        energy.append(torch.vdot(lam, mu).real.item())
        row = []
        for op in reversed(ops):
            if op.params:
                g = _apply(lam.clone(), n, _PAULI["Pauli" + op.name[1]], op.wires)
                row.append(torch.vdot(mu, g).imag)
            _apply_op(lam, n, op, True)
            _apply_op(mu, n, op, True)
        jac.append(torch.stack(row[::-1]).cpu().numpy())
    return np.array(energy), np.concatenate(jac)


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "serve":
        reqs = _requests(case, seed)
        if sum(4.0 * len(r.ops) + 3.0 * 50 for r in reqs) > 200000:
            return None
        got = [_gradient(r.ops, r.n, _run_exact(r.ops, r.n, device), [(r.coeffs, r.words)]) for r in reqs]
        return {"energies": np.concatenate([e for e, _ in got]), "gradients": np.concatenate([g for _, g in got])}
    n = case["n"]
    if kind == "circuit":
        ops = _circuit_ops(case, seed, False)
        if len(ops) * 2.0 ** n > 2e11:
            return None
        if case["bits"] == 64:
            for op in ops:
                if op.matrix is not None:  # the entry point takes single-precision matrices
                    op.matrix = op.matrix.astype(np.complex64)
        psi = _run_exact(ops, n, device)
        if case["result"] == "state":
            return {"state": psi}
        p = [_marginal(psi, n, [w]) for w in range(n)]
        out = {"z": np.array([v[0] - v[1] for v in p])}
        if case["result"] == "probs":
            out["probs"] = _marginal(psi, n, list(range(min(n, 10))))
        return out
    if kind == "gradient":
        ops = _circuit_ops(case, seed, True)
        energy, jac = _gradient(ops, n, _run_exact(ops, n, device), _pauli_sums(case, seed))
        return {"jacobian": jac, "energy": energy}
    if kind == "training":
        ops = _circuit_ops(case, seed, True)
        psi = _run_exact(ops, n, device)
        words = [[[(("PauliX", "PauliY", "PauliZ")[k % 3], (5 * k) % n)]] for k in range(case["observables"])]
        ev = np.array([torch.vdot(psi, _apply_sum(psi, n, [1.0], w)).real.item() for w in words])
        _, grad = _gradient(ops, n, psi, [(list(2 * ev), [w[0] for w in words])])
        return {"expvals": torch.from_numpy(ev), "gradient": torch.from_numpy(grad)}
    psi = _random_state(n, seed, device).to(_state_dtype(case)).to(torch.complex128)
    if kind == "matrix":
        for mat, wires, ctrls, values, inverse in _matrix_ops(case, seed):
            mat = mat.astype(np.complex64 if case["bits"] == 64 else np.complex128)
            _apply(psi, n, mat.conj().T if inverse else mat, wires, ctrls, values)
        return {"state": psi}
    wires, pair, herm, (coeffs, words) = _measure_inputs(case, seed)
    if case["bits"] == 64:
        herm = herm.astype(np.complex64)
    mean = lambda v: torch.vdot(psi, v).real.item()  # noqa: E731
    h = _apply_sum(psi, n, [1.0], words[:1])
    out = {"probs": _marginal(psi, n, wires), "energy": mean(_apply_sum(psi, n, coeffs, words)),
           "x": mean(_apply(psi.clone(), n, _X, pair[:1])), "hermitian": mean(_apply(psi.clone(), n, herm, pair)),
           "variance": torch.vdot(h, h).real.item() - mean(h) ** 2}
    if case["shots"]:
        out["samples"] = None
    return out
