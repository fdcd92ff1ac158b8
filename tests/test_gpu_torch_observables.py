"""Several one-wire observables of one differentiable circuit: wires out of
range are refused as they are one at a time, and the identity's mean is the
squared norm of the state."""
import numpy as np
import pytest

from helpers import TOL_C128, oracle_run
from oracle import lq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
T = pytest.importorskip("lightning_amd.torch_interface")
W = pytest.importorskip("lightning_amd.workloads")
L = pytest.importorskip("lightning_amd.lightning_qubit_ops")


def circuit(n):
    return [W.CircuitOp("RX", [w], [0.3 + w]) for w in range(n)] + [W.CircuitOp("CNOT", [w, w + 1]) for w in range(n - 1)]


def params(ops):
    return torch.tensor([p for o in ops for p in o.params], dtype=torch.float64)


@pytest.mark.parametrize("bits", [128, 64])
@pytest.mark.parametrize("name", ["Identity", "PauliZ", "Hadamard"])
def test_wires_out_of_range_are_refused(bits, name):
    ops = circuit(4)
    with pytest.raises(L.LightningException, match="observable wire out of range"):
        T.circuit_expvals(params(ops), 4, ops, [("N", "PauliX", 0), ("N", name, 4)], bits)


def test_identity_is_the_norm():
    n = 5
    ops = circuit(n) + [W.CircuitOp("QubitUnitary", [2], [], matrix=np.array([[0.5, 0.1], [0.2j, 0.8]]))]
    psi = oracle_run(n, ops)
    got = T.circuit_expvals(params(ops), n, ops, [("N", "Identity", 1), ("N", "PauliZ", 3)]).numpy()
    np.testing.assert_allclose(got, [np.vdot(psi, psi).real, O.expval_named(psi, n, "PauliZ", [3])], rtol=0, atol=TOL_C128)
