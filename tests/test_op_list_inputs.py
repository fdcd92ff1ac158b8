"""Op lists given as iterators, wire lists given as iterators and bytes, the
lists that an OpsStruct gives back, and bound copies of ops that are not plain
CircuitOps."""
import pytest

from lightning_amd import lightning_qubit_ops as L
from lightning_amd import workloads as W
from lightning_amd._capi import u32


@pytest.mark.parametrize("values,expected", [(lambda: (float(i) for i in (1, 2, 3)), [1, 2, 3]),
                                             (lambda: (i for i in ()), []), (lambda: b"\0\1\2\3", [0, 1, 2, 3]),
                                             (lambda: bytearray(b"\0\1\2\3"), [0, 1, 2, 3]), (lambda: {3: 1}, [3])])
def test_wire_iterators_and_bytes(values, expected):
    a, p, n = u32(values())
    assert [p[i] for i in range(n)] == expected
