"""Tile passes planned and run in host memory: the planner of
qcsim_amd/csrc/circuit_plan.cpp with tests/cpp/circuit_host.cpp, which states
in C++ what each operation of a pass does, against the oracle."""
import ctypes as C
import os
import subprocess
import time

import numpy as np
import pytest

from gatecatalog import catalog
from qcsim_amd import QubitRegister
from qcsim_amd import gates as G
from qcsim_amd._lib import QcsGate
from refmath import random_state
from test_gpu_circuit import circuit, ladder, run_oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STREAM = 64 * 64 * 8 - 256  # a register's staging slot, less its rounding


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("plan") / "libcircuit_host.so")
    src = [os.path.join(ROOT, p) for p in ("tests/cpp/circuit_host.cpp", "qcsim_amd/csrc/circuit_plan.cpp",
                                          "qcsim_amd/csrc/fusion.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"),
                    *src, "-o", lib], check=True)
    L = C.CDLL(lib)
    L.plan_new.restype, L.plan_new.argtypes = C.c_void_p, [C.c_void_p, C.c_uint32, C.c_uint32, C.c_uint64, C.c_uint64]
    L.plan_free.restype, L.plan_free.argtypes = None, [C.c_void_p]
    L.plan_width.restype, L.plan_width.argtypes = C.c_uint32, [C.c_void_p, *[C.c_uint32] * 2, *[C.c_uint64] * 2,
                                                               *[C.c_uint32] * 2]
    L.plan_step.restype = C.c_int64
    L.plan_step.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.POINTER(C.c_uint64)]
    return L


def steps(host, arr, count, nq, amp_bytes=16, stream=STREAM, psi=None, single=None):
    """(passes, gates by themselves, the longest stream); psi is updated in place."""
    plan = host.plan_new(arr, count, nq, amp_bytes, stream)
    passes, alone, longest = 0, 0, 0
    nbytes = C.c_uint64()
    while True:
        k = host.plan_step(plan, arr, nq, None if psi is None else psi.ctypes.data, C.byref(nbytes))
        if k == -1:
            break
        if k == -2:
            passes += 1
            longest = max(longest, nbytes.value)
        else:
            alone += 1
            if single:
                single(int(k))
    host.plan_free(plan)
    return passes, alone, longest


def run_planned(host, psi, n, seq, **kw):
    out = np.ascontiguousarray(psi, dtype=np.complex128).copy()

    def single(k):
        out[:] = run_oracle(out, n, [seq[k]])

    return out, steps(host, QubitRegister._gate_array(seq), len(seq), n, psi=out, single=single, **kw)


# amp_bytes 8192: as for a register above 64 MiB, whose few gates launch by themselves
@pytest.mark.parametrize("amp_bytes", [16, 8, 8192])
@pytest.mark.parametrize("n,blocks", [(3, False), (4, True), (5, False), (9, False), (10, True), (11, False), (13, True),
                                      (14, False)])
def test_passes_equal_oracle(host, n, blocks, amp_bytes):
    rng = np.random.default_rng(1000 * n + amp_bytes)
    psi = random_state(rng, n)
    seq = circuit(rng, n, blocks)
    got, (passes, alone, longest) = run_planned(host, psi, n, seq, amp_bytes=amp_bytes)
    assert np.max(np.abs(got - run_oracle(psi, n, seq))) < 1e-12
    assert passes and longest <= STREAM + 256 and alone >= 2 * blocks * (n >= 5)


@pytest.mark.parametrize("stream", [2048, 4096])
def test_passes_keep_to_the_stream(host, stream):
    """A short staging slot makes more passes, none longer than it."""
    n = 7
    rng = np.random.default_rng(stream)
    psi = random_state(rng, n)
    seq = circuit(rng, n, False)
    got, (passes, _, longest) = run_planned(host, psi, n, seq, stream=stream)
    assert np.max(np.abs(got - run_oracle(psi, n, seq))) < 1e-12
    assert passes > 2 and longest <= stream + 256


@pytest.mark.parametrize("n", [4, 12])
def test_long_lists(host, n):
    """More gates than the planner takes in at once, with ladders across the
    places where it goes on."""
    rng = np.random.default_rng(n)
    one, two, three = catalog(n)
    fams = one + two + three
    seq = []
    while len(seq) < 5000:
        seq += ladder(rng, n)
        _, gate = fams[int(rng.integers(len(fams)))]
        seq.append((gate, [int(x) for x in rng.choice(n, size=gate.getQubitsNumber(), replace=False)]))
    psi = random_state(rng, n)
    got, _ = run_planned(host, psi, n, seq)
    assert np.max(np.abs(got - run_oracle(psi, n, seq))) < 1e-12


def test_planning_grows_with_the_list(host):
    """Ising steps on few qubits, each CNOT, Rz, CNOT one gate to the planner.
    The time of the whole plan is proportional to the list, and that of its
    first pass does not depend on it (a factor of five left for the clock)."""
    n, rng = 4, np.random.default_rng(1)
    seq = []
    while len(seq) < 2000:
        q = int(rng.integers(n - 1))
        seq += [(G.CNOTGate(), [q + 1, q]), (G.RzGate(0.1), [q + 1]), (G.CNOTGate(), [q + 1, q])]
        seq.append((G.RxGate(0.2), [int(rng.integers(n))]))
    long = 32
    arr = (QcsGate * (long * len(seq)))()
    one = QubitRegister._gate_array(seq)
    head = 32 + 2 * 16 * 8  # header and a 4 x 4 matrix; the rest of a gate stays untouched
    for r in range(long):
        for i in range(len(seq)):
            C.memmove(C.byref(arr[r * len(seq) + i]), C.byref(one[i]), head)

    def best(count, first):
        times = []
        for _ in range(5):
            t = time.perf_counter()
            if first:
                plan = host.plan_new(arr, count, n, 16, STREAM)
                assert host.plan_step(plan, arr, n, None, C.byref(C.c_uint64())) == -2
                host.plan_free(plan)
            else:
                steps(host, arr, count, n)
            times.append(time.perf_counter() - t)
        return min(times)

    assert best(long * len(seq), False) < 5 * long * best(len(seq), False)
    assert best(long * len(seq), True) < 5 * best(len(seq), True)


def layers(n, rng):
    seq = []
    for _ in range(10):
        seq += [(G.SingleQubitGate(G.haar_u2(rng)), [q]) for q in range(n)]
        perm = [int(q) for q in rng.permutation(n)]
        seq += [(G.CNOTGate(), [a, b]) for a, b in zip(perm[0::2], perm[1::2])]
    return seq


def ising_steps(n):
    seq = []
    for _ in range(5):
        for q in range(n - 1):
            seq += [(G.CNOTGate(), [q + 1, q]), (G.RzGate(0.2), [q + 1]), (G.CNOTGate(), [q + 1, q])]
        seq += [(G.RxGate(0.3), [q]) for q in range(n)]
    return seq


def heisenberg_steps(n):
    seq = []
    for _ in range(3):
        for q in [*range(0, n - 1, 2), *range(1, n - 1, 2)]:
            for before, after in ((G.HadamardGate(), G.HadamardGate()), (G.RxGate(1.5), G.RxGate(-1.5)), (None, None)):
                seq += [(before, [q]), (before, [q + 1])] if before else []
                seq += [(G.CNOTGate(), [q + 1, q]), (G.RzGate(0.2), [q + 1]), (G.CNOTGate(), [q + 1, q])]
                seq += [(after, [q]), (after, [q + 1])] if after else []
    return seq


# what the rule says where both ways were timed, and next to where it begins
@pytest.mark.parametrize("amp_bytes,n,kind,width,blocks", [
    (16, 24, "heisenberg", 5, False), (16, 26, "heisenberg", 5, True), (16, 27, "heisenberg", 4, True),
    (16, 28, "heisenberg", 5, True), (16, 26, "layers", 4, False), (16, 28, "layers", 5, False),
    (16, 28, "ising", 5, False), (16, 28, "heisenberg", 3, False), (8, 27, "heisenberg", 5, False),
    (8, 28, "heisenberg", 5, True), (8, 28, "heisenberg", 4, True), (8, 28, "layers", 5, True), (8, 30, "layers", 4, True),
    (8, 28, "ising", 4, False), (8, 30, "ising", 4, False), (8, 28, "ising", 3, False)])
def test_blocks_or_passes(host, amp_bytes, n, kind, width, blocks):
    seq = {"layers": lambda: layers(n, np.random.default_rng(n)), "ising": lambda: ising_steps(n),
           "heisenberg": lambda: heisenberg_steps(n)}[kind]()
    arr = QubitRegister._gate_array(seq)
    assert host.plan_width(arr, len(seq), n, amp_bytes, STREAM, width, width) == (width if blocks else 0)
    picked = host.plan_width(arr, len(seq), n, amp_bytes, STREAM, 2, 5)
    assert picked in (4, 5) if blocks else width < 4 or picked == 0
    assert host.plan_width(arr, 0, n, amp_bytes, STREAM, 2, 5) in (0, 4, 5)  # an empty list
