"""What a gate call takes for its matrix (no device: the library refuses a
null register before it reads anything)."""
import ctypes as C

import numpy as np
import pytest

from qcsim_amd import QubitRegister
from qcsim_amd._lib import lib
from qcsim_amd.register import _mat_bytes


class Nested:
    """A gate that keeps its matrix as nested lists."""

    traits = 0

    def __init__(self, m):
        self.m = m

    def getQubitsNumber(self):
        return 1

    def getRawOperatorMatrix(self):
        return self.m


@pytest.mark.parametrize("m", [[[0, 1], [1, 0]], ((0, 1j), (-1j, 0)), np.eye(2), np.eye(2, dtype=np.complex64),
                               np.array([[1, 2], [3, 4j]]).T])
def test_a_matrix_of_any_form_reaches_the_library(m):
    assert _mat_bytes(m) == np.array(m, dtype=np.complex128).tobytes()
    reg = QubitRegister.__new__(QubitRegister)
    reg._h, reg._record = None, False
    with pytest.raises(ValueError, match="null"):
        reg.ApplyGate(Nested(m), 0)


def test_the_matrix_argument_is_doubles_or_bytes():
    m = np.eye(2, dtype=np.complex128)
    for ok in (m.tobytes(), m.ctypes.data_as(C.POINTER(C.c_double)), (C.c_double * 8)(), None):
        assert lib().qcs_apply_gate(None, 1, 0, 0, 0, 0, ok) != 0
    for bad in ("text", 4096, 1.0, m, (C.c_float * 8)()):
        with pytest.raises(C.ArgumentError):
            lib().qcs_apply_gate(None, 1, 0, 0, 0, 0, bad)
