"""Op lists given as iterators, wire lists given as iterators and bytes, the
lists that an OpsStruct gives back, and bound copies of ops that are not plain
CircuitOps."""
import pytest

from lightning_amd import lightning_qubit_ops as L
from lightning_amd import workloads as W
from lightning_amd._capi import u32


@pytest.mark.parametrize("rows", [lambda v: (x for x in v), lambda v: map(tuple, v), lambda v: [iter(x) for x in v]])
def test_ops_struct_from_iterators(rows):
    ops = L.OpsStructC128(["RX", "CRY"], rows([[0.1], [0.2]]), rows([[0], [1]]), iter([False, True]), iter([[], []]),
                          rows([[], [2]]), rows([[], [True]]))
    assert ops.params == [[0.1], [0.2]] and ops.wires == [[0], [1]] and ops.inverses == [False, True]
    assert ops.ctrl_wires == [[], [2]] and ops.ctrl_values == [[], [True]]


def test_ops_struct_lists_are_attributes():
    ops = L.OpsStructC128(["RX"], [[0.1]], [[0]], [False], [[]])
    ops.params = [[5.0]]
    ops.wires.append([3])
    assert ops.params == [[5.0]] and ops.wires == [[0], [3]]
    assert ops.ctrl_wires is ops.ctrl_wires and ops.ctrl_values is ops.ctrl_values


@pytest.mark.parametrize("values,expected", [(lambda: (float(i) for i in (1, 2, 3)), [1, 2, 3]),
                                             (lambda: (i for i in ()), []), (lambda: b"\0\1\2\3", [0, 1, 2, 3]),
                                             (lambda: bytearray(b"\0\1\2\3"), [0, 1, 2, 3]), (lambda: {3: 1}, [3])])
def test_wire_iterators_and_bytes(values, expected):
    a, p, n = u32(values())
    assert [p[i] for i in range(n)] == expected


def test_gate_lists_without_length_are_refused():
    sv = object.__new__(L.StateVectorC128)
    for wires, params in (([iter([0])], [[0.1]]), ([[0]], [iter([0.1])])):
        with pytest.raises(TypeError):
            sv.applyOperations(["RX"], wires, [False], params)


def test_bind_takes_any_op():
    T = pytest.importorskip("lightning_amd.torch_interface")

    class Op:
        name, wires, params, inverse, matrix, ctrls, cvals = "RX", [0], [0.1], False, None, [], []

    class Derived(W.CircuitOp):
        pass

    expected = W.CircuitOp("RX", [0], [0.7])
    for op in (Op(), Derived("RX", [0], [0.1]), W.CircuitOp("RX", [0], [0.1])):
        assert T.bind([op], [0.7]) == [expected]
