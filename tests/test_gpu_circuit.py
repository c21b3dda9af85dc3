"""Circuits in tile passes against the oracle: every gate family with its
qubits inside and outside a tile, where tiles begin (3 qubits), fill a
register (10), leave one and more qubits outside (11..20), and the CNOT
ladders that the planner takes together."""
import numpy as np
import pytest

from gatecatalog import catalog
from oracle.oracle import OracleRegister
from qcsim_amd import QubitRegister
from qcsim_amd import gates as G
from refmath import random_state, random_unitary

pytestmark = pytest.mark.gpu


class Block:
    """A dense block of four or five qubits: no tile operation."""

    traits, flags = 0, 1

    def __init__(self, m):
        self.m = m

    def getQubitsNumber(self):
        return self.m.shape[0].bit_length() - 1

    def getRawOperatorMatrix(self):
        return self.m


def ladder(rng, n):
    """exp(i phi Z..Z) as CNOTs around an Rz, with gates on other qubits, and
    sometimes on the ladder's own, in between."""
    q = [int(x) for x in rng.permutation(n)[: int(rng.integers(2, min(n, 6) + 1))]]
    down = [(G.CNOTGate(), [b, a]) for a, b in zip(q, q[1:])]
    mid = [(G.RzGate(float(rng.uniform(-3, 3))), [q[-1]])]
    if rng.integers(3) == 0:
        mid.insert(int(rng.integers(2)), (G.RyGate(0.7), [int(rng.integers(n))]))
    up = down[::-1]
    if rng.integers(3) == 0:
        up.insert(int(rng.integers(len(up))), (G.PhaseShiftGate(0.3), [int(rng.integers(n))]))
    return down + mid + up


def circuit(rng, n, blocks):
    seq = []
    for fam in (f for k in catalog(n) for f in k):
        k = fam[1].getQubitsNumber()
        for _ in range(2):
            seq.append((fam[1], [int(x) for x in rng.choice(n, size=k, replace=False)]))
    seq = [seq[i] for i in rng.permutation(len(seq))]
    for at in sorted(rng.integers(0, len(seq), 8), reverse=True):
        seq[at:at] = ladder(rng, n)
    for k in (4, 5) if blocks else ():
        if n >= k:
            at = int(rng.integers(len(seq)))
            seq.insert(at, (Block(random_unitary(rng, 1 << k)), [int(x) for x in rng.permutation(n)[:k]]))
    return seq


def run_oracle(psi, n, seq):
    o = OracleRegister(n)
    o.set_state(psi)
    for gate, qs in seq:
        if isinstance(gate, Block):
            o.apply_dense(qs, gate.m)
        else:
            o.apply_gate(gate, *qs)
    return o.state()


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,blocks", [(3, False), (4, True), (9, False), (10, True), (11, False), (13, True),
                                      (18, False), (19, False), (20, False)])
def test_circuit_equals_oracle(n, blocks, precision):
    rng = np.random.default_rng(100 * n + blocks)
    psi = random_state(rng, n)
    seq = circuit(rng, n, blocks)
    want = run_oracle(psi, n, seq)
    g = QubitRegister(n, precision=precision)
    g.setRegisterStorageFastNoNormalize(psi.copy())
    g.apply_circuit(seq)
    got = np.asarray(g.getRegisterStorage())
    g.close()
    if precision == "c128":
        assert np.max(np.abs(got - want)) < 1e-12
    else:  # one rounding of each part a pass, some more in a block's own FP32 kernel
        assert np.linalg.norm(got - want) < 4 * len(seq) * 2.0**-24 * np.linalg.norm(want)


@pytest.mark.parametrize("width", [2, 5, "auto"])
def test_refused_gate_ends_the_circuit(width):
    """A gate whose qubits repeat is refused by its entry point; in a circuit
    of width 0 the gates before it have been applied."""
    n = 11
    psi = random_state(np.random.default_rng(7), n)
    seq = [(G.HadamardGate(), [3]), (G.CNOTGate(), [10, 3]), (G.CNOTGate(), [4, 4]), (G.HadamardGate(), [0])]
    g = QubitRegister(n)
    g.setRegisterStorageFastNoNormalize(psi.copy())
    with pytest.raises(Exception):
        g.apply_circuit(seq)
    assert np.max(np.abs(g.getRegisterStorage() - run_oracle(psi, n, seq[:2]))) < 1e-12
    g.setRegisterStorageFastNoNormalize(psi.copy())
    with pytest.raises(Exception):
        g.apply_circuit([(G.HadamardGate(), [3]), (G.HadamardGate(), [n])], fuse_width=width)
    assert np.array_equal(g.getRegisterStorage(), psi)
    g.close()


@pytest.mark.parametrize("n", [3, 6, 12, 16, 23])
@pytest.mark.parametrize("count", [1, 2, 3])
def test_few_gates(n, count):
    """Lists too short for a pass, of which a CNOT, Rz, CNOT in the middle is
    one gate to the planner and has no launch of its own: on registers of one
    tile, of several and above 64 MiB."""
    rng = np.random.default_rng(10 * n + count)
    psi = random_state(rng, n)
    for k in range(4):
        a, b, c = (int(x) for x in rng.permutation(n)[:3])
        seq = [(G.CNOTGate(), [a, b]), (G.RzGate(0.7 + k), [a]), (G.CNOTGate(), [a, b])]
        if k & 1:
            seq += [(G.CNOTGate(), [b, c]), (G.RzGate(0.4), [b]), (G.CNOTGate(), [b, c])]
        if k & 2:
            seq.insert(int(rng.integers(len(seq))), (G.RyGate(0.3), [c]))
        seq = seq * (count - 1) + seq
        g = QubitRegister(n)
        g.setRegisterStorageFastNoNormalize(psi.copy())
        g.apply_circuit(seq)
        got = np.asarray(g.getRegisterStorage())
        g.close()
        assert np.max(np.abs(got - run_oracle(psi, n, seq))) < 1e-12, k


@pytest.mark.parametrize("n,width", [(27, 5), (28, 4), (28, 5), (28, "auto")])
def test_large_complex64_circuit_and_its_inverse(n, width):
    """Where complex64 circuits go over to dense blocks: a list fused to the
    width, then as a program with the inverse order, from |0> back to |0>. An
    FP32 block of 32 rows errs by at most 32 * 6e-8 of an amplitude and the 30
    gates make at most 12 blocks each way: 5e-5."""
    rng = np.random.default_rng(n)
    seq = [(G.SingleQubitGate(G.haar_u2(rng)), [int(q)]) for q in rng.permutation(n)[:20]]
    for at in sorted(rng.integers(0, 20, 10), reverse=True):
        seq.insert(int(at), (G.CNOTGate(), [int(q) for q in rng.choice(n, 2, replace=False)]))
    g = QubitRegister(n, precision="c64")
    g.setToBasisState(0)
    g.apply_circuit(seq, width)
    prog = g.compile_program(seq, width, adjoint=True)
    prog.run()
    amp = g.getBasisStateAmplitude(0)
    prog.close()
    g.close()
    assert abs(amp - 1) < 5e-5
