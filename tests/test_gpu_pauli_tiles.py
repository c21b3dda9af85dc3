"""Pauli strings in tile passes: registers around a tile (1..14 qubits), x masks
inside one tile, across two, on its register qubits and too wide for any, z
masks inside and outside, more masks than a pass has slots and more terms
than it has results."""
import numpy as np
import pytest

from qcsim_amd import QubitRegister
from qcsim_amd import gates as G
from refmath import random_state

pytestmark = pytest.mark.gpu


def reference(psi, x, z):
    s = np.arange(psi.size, dtype=np.uint64)
    sign = 1.0 - 2.0 * (np.bitwise_count(s & np.uint64(z)) & 1)
    ny = bin(x & z).count("1")
    # (P psi)_{s ^ x} = i^ny (-1)^{popcount(s & z)} psi_s
    return float(np.real(1j**ny * np.sum(np.conj(psi[s ^ np.uint64(x)]) * sign * psi)))


def masks(kind, n, rng):
    full = (1 << n) - 1
    if kind == "chain":
        x = [3 << q for q in range(n - 1)]
        return [(v, w) for v in x for w in (0, v)] + [(0, v) for v in x] + [(0, 1 << q) for q in range(n)]
    if kind == "diagonal":  # more than a pass's slots for masks that leave the tile
        return [(0, int(z)) for z in rng.integers(0, full + 1, 70)] + [(0, 1 << q) for q in range(n)]
    if kind == "dense":  # few x masks, many z masks
        xs = [int(v) for v in rng.integers(0, full + 1, 5)] + [full, 1, 1 << (n - 1)]
        return [(xs[i % len(xs)], int(z)) for i, z in enumerate(rng.integers(0, full + 1, 150))]
    pairs = [(1 << a) | (1 << b) for a in range(n) for b in range(a)] + [1 << q for q in range(n)]
    return [(x, int(rng.integers(0, full + 1))) for x in pairs]


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 12, 13, 14])
@pytest.mark.parametrize("kind", ["chain", "diagonal", "dense", "pairs"])
def test_terms_equal_reference(kind, n, precision):
    rng = np.random.default_rng(1000 + n)
    g = QubitRegister(n, precision=precision)
    g.setRegisterStorageFastNoNormalize(random_state(rng, n))
    psi = np.asarray(g.getRegisterStorage()).astype(np.complex128)
    terms = masks(kind, n, rng)
    got = g.pauli_expectation([x for x, _ in terms], [z for _, z in terms])
    g.close()
    want = np.array([reference(psi, x, z) for x, z in terms])
    # sums of 2^n products in FP64 whatever the state's type
    assert np.max(np.abs(got - want)) < 1e-13


@pytest.mark.parametrize("count", [1, 9, 10, 17])
def test_terms_of_one_x_mask_on_a_large_state(count):
    """Above 256 MiB, terms that share an x mask but no z bits outside a tile
    leave the tile passes from some number on: together and one by one, which
    always is a tile pass, they are the same FP64 sums in another order."""
    rng = np.random.default_rng(count)
    g = QubitRegister(25)
    g.setToEqualSuperposition()
    for q in range(25):
        g.ApplyGate(G.SingleQubitGate(G.haar_u2(rng)), q)
    x = [3 << 11] * count + [1]
    z = [int(v) for v in rng.integers(0, 1 << 25, count + 1)]
    got = g.pauli_expectation(x, z)
    want = [float(g.pauli_expectation([a], [b])[0]) for a, b in zip(x, z)]
    g.close()
    assert np.max(np.abs(got - np.array(want))) < 1e-13
