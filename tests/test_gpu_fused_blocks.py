"""Gate lists at a fusion width on the device."""
import ctypes as C

import numpy as np
import pytest

from qcsim_amd import QubitRegister, _lib
from qcsim_amd import gates as G

pytestmark = pytest.mark.gpu


def test_auto_without_a_cost_table():
    """QCS_FUSE_AUTO neither measures nor fuses where a list runs in passes:
    the state equals width 0's bit for bit, and no width is reported."""
    n = 17
    rng = np.random.default_rng(1)
    seq = [(G.SingleQubitGate(G.haar_u2(rng)), [q]) for _ in range(4) for q in range(n)]
    seq += [(G.CNOTGate(), [q + 1, q]) for q in range(n - 1)]
    costs = np.zeros(6)
    pd = C.POINTER(C.c_double)
    for p in ("c128", "c64"):
        a, b = QubitRegister(n, precision=p), QubitRegister(n, precision=p)
        prec = {"c128": _lib.QCS_COMPLEX128, "c64": _lib.QCS_COMPLEX64}[p]
        _lib.check(_lib.lib().qcs_set_fusion_costs(prec, n, np.zeros(6).ctypes.data_as(pd)))
        before = a.launch_count()
        a.apply_circuit(seq, fuse_width="auto")
        launches = a.launch_count() - before
        before = b.launch_count()
        b.apply_circuit(seq)
        assert launches == b.launch_count() - before
        assert a.last_fuse_width() == 0
        _lib.check(_lib.lib().qcs_get_fusion_costs(prec, n, costs.ctypes.data_as(pd)))
        assert not costs.any()
        prog = b.compile_program(seq, fuse_width="auto")
        b.setToBasisState(0)
        prog.run()
        assert np.array_equal(a.getRegisterStorage(), b.getRegisterStorage())
        prog.close()
        a.close()
        b.close()
