"""Gate lists at a fusion width on the device: those that run in dense blocks
against the same lists in tile passes, where registers are large enough for
it."""
import ctypes as C

import numpy as np
import pytest

from qcsim_amd import QubitRegister, _lib
from test_circuit_plan import heisenberg_steps, ising_steps, layers
from test_fusion import to_struct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,kind,width,blocks", [
    (25, "c128", "heisenberg", 4, True), (26, "c128", "heisenberg", 5, True), (26, "c128", "heisenberg", "auto", True),
    (25, "c128", "layers", 5, False), (27, "c64", "heisenberg", 5, False), (28, "c64", "heisenberg", 4, True),
    (28, "c64", "layers", 5, True), (28, "c64", "layers", "auto", True), (28, "c64", "ising", 4, False)])
def test_list_in_blocks_equals_passes(n, precision, kind, width, blocks):
    """The whole state of a list at a fusion width against width 0, which is
    always tile passes, and how many launches it took. In complex64 the two
    differ by what FP32 blocks of 2^5 rows may err, a row
    34 2^-24 of its vector's norm."""
    seq = {"layers": lambda: layers(n, np.random.default_rng(n)), "ising": lambda: ising_steps(n),
           "heisenberg": lambda: heisenberg_steps(n)}[kind]()
    a, b = QubitRegister(n, precision=precision), QubitRegister(n, precision=precision)
    for r in (a, b):
        r.setToBasisState(5)
    before = a.launch_count()
    a.apply_circuit(seq, fuse_width=width)
    launches = a.launch_count() - before
    b.apply_circuit(seq)
    if blocks:
        w = a.last_fuse_width()
        assert w == width or width == "auto" and w in (4, 5)
        out = (_lib.QcsGate * len(seq))()
        count = C.c_uint32()
        _lib.check(_lib.lib().qcs_fuse(to_struct(seq), len(seq), w, out, C.byref(count)))
        assert launches == count.value
    else:
        assert launches < len(seq) / 10
    largest, overlap = a.compare(b)
    na, nb = a.norm2(), b.norm2()
    a.close()
    b.close()
    if precision == "c128":
        assert largest < 1e-12
    else:
        tol = 60 * 34 * 2 * 2.0**-24  # at most 60 blocks
        assert 1 - abs(overlap) ** 2 / (na * nb) < tol**2 + 1e-12
        assert abs(na - 1) < 2 * tol and abs(nb - 1) < 2 * tol


def test_auto_without_a_cost_table():
    """QCS_FUSE_AUTO neither measures nor fuses where a list runs in passes:
    the state equals width 0's bit for bit, and no width is reported."""
    n = 17
    seq = layers(n, np.random.default_rng(1))
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
