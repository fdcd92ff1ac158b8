"""Op lists cross the binding as flat arrays: what the Python classes accept
and give back (lists, tuples, numpy scalars, missing controls, matrices), and
that short lists are refused before the library sees them."""
import numpy as np
import pytest

from lightning_amd import lightning_qubit_ops as L
from lightning_amd import workloads as W
from lightning_amd._capi import u32


def test_ops_struct_fields():
    ops = L.OpsStructC128(["RX", "CNOT", "QubitUnitary", "RY"], [(0.3,), [], [0.0], [np.float32(0.5)]],
                          [[0], (0, 1), np.array([2]), [np.int64(3)]], [False, True, 0, np.True_],
                          [[], None, np.eye(2), []], [[], [], [], [1]], [[], [], [], [np.True_]])
    assert ops.params == [[0.3], [], [0.0], [0.5]]
    assert ops.wires == [[0], [0, 1], [2], [3]]
    assert ops.inverses == [False, True, False, True]
    assert ops.ctrl_wires == [[], [], [], [1]] and ops.ctrl_values == [[], [], [], [True]]
    assert [m.shape for m in ops.matrices] == [(0,), (0,), (4,), (0,)]
    assert ops.getNumParOps() == 3 and repr(ops) == "Operations: [RX, CNOT, QubitUnitary, RY]"
    assert W.to_ops([]).getNumParOps() == 0
    float_wires = L.OpsStructC64(["RZ"], [[1]], [[2.0]], [False], [[]])
    assert float_wires.wires == [[2]] and float_wires.params == [[1.0]]


def test_short_lists_are_refused():
    with pytest.raises(IndexError):
        L.OpsStructC128(["RX", "RY"], [[0.1]], [[0], [1]], [False, False], [[], []])
    with pytest.raises(IndexError):
        L.OpsStructC128(["RX", "RY"], [[0.1], [0.2]], [[0]], [False, False], [[], []])
    with pytest.raises(OverflowError):
        L.OpsStructC128(["RX"], [[0.1]], [[-1]], [False], [[]])


@pytest.mark.parametrize("values,expected", [([1, 2], [1, 2]), (np.array([3, 4]), [3, 4]), (np.array([1.0, 2.0]), [1, 2]),
                                             (range(3), [0, 1, 2]), ((), []), ([[1, 2]], [1, 2])])
def test_wire_arrays(values, expected):
    a, p, n = u32(values)
    assert n == len(expected) and [p[i] for i in range(n)] == expected
