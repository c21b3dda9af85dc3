"""The blocks of the fusion pass on the device: every width's blocks one by one
against the oracle on small registers, and gate lists that run in blocks
against the same lists in tile passes where registers are large enough for
it."""
import ctypes as C

import numpy as np
import pytest

from oracle.oracle import OracleRegister
from qcsim_amd import QubitRegister, _lib
from refmath import random_state
from test_circuit_plan import heisenberg_steps, ising_steps, layers
from test_fusion import fuse, random_circuit, to_struct

pytestmark = pytest.mark.gpu


def apply_block(reg, g):
    m = np.frombuffer(bytes(g.mat), dtype=np.float64)[: 2 * 4**g.k].view(np.complex128).reshape(1 << g.k, 1 << g.k)
    if (g.flags & _lib.QCS_GATE_DENSE) or g.k > 3:
        reg.apply_dense([g.qubits[j] for j in range(g.k)], m)
    else:
        _lib.check(_lib.lib().qcs_apply_gate(reg._h, g.k, g.traits, *g.qubits[:3], m.tobytes()))


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("width", [2, 3, 4, 5])
@pytest.mark.parametrize("n", [5, 7, 9, 13])
def test_blocks_equal_oracle(n, width, precision):
    """n = 5, 7: states below one tile of the matrix-core kernel. In complex64 a
    row of a block errs by at most (2^k + 2) 2^-24 of its vector's norm."""
    rng = np.random.default_rng(10 * n + width)
    seq = random_circuit(rng, n, 80)
    psi = random_state(rng, n)
    ref = OracleRegister(n)
    ref.set_state(psi)
    for gate, qs in seq:
        ref.apply_gate(gate, *qs)
    out, count = fuse(to_struct(seq), width)
    assert any(out[i].flags & _lib.QCS_GATE_DENSE for i in range(count))
    reg = QubitRegister(n, precision=precision)
    reg.setRegisterStorageFastNoNormalize(psi.copy())
    for i in range(count):
        apply_block(reg, out[i])
    err = np.asarray(reg.getRegisterStorage()) - ref.state()
    reg.close()
    if precision == "c128":
        assert np.max(np.abs(err)) < 1e-12
    else:
        assert np.linalg.norm(err) < count * (2**width + 2) * 2 * 2.0**-24


@pytest.mark.parametrize("n,precision,kind,width,blocks", [
    (25, "c128", "heisenberg", 4, True), (26, "c128", "heisenberg", 5, True), (26, "c128", "heisenberg", "auto", True),
    (25, "c128", "layers", 5, False), (27, "c64", "heisenberg", 5, False), (28, "c64", "heisenberg", 4, True),
    (28, "c64", "layers", 5, True), (28, "c64", "layers", "auto", True), (28, "c64", "ising", 4, False)])
def test_list_in_blocks_equals_passes(n, precision, kind, width, blocks):
    """The whole state of a list at a fusion width against width 0, which is
    always tile passes, and how many launches it took. In complex64 the two
    differ by what FP32 blocks of 2^5 rows may err, as above."""
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
    if blocks:  # a program of the list takes the same blocks
        prog = b.compile_program(seq, fuse_width=width)
        b.setToBasisState(5)
        prog.run()
        assert prog.launches() == count.value and a.compare(b)[0] == 0
        prog.close()
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
