"""Batched VQE at the edges of its work units: one to five instances a wave
each, sizes around the largest of a wave (10) and the padded ones (1..4),
partial layers, more layers than one table of rotations holds, and more terms
than a wave holds at once."""
import math

import numpy as np
import pytest

from oracle.oracle import OracleRegister
from qcsim_amd.vqe import VqeBatch, ansatz_gates

pytestmark = pytest.mark.gpu


def exact(n, params, xs, zs, cs):
    o = OracleRegister(n)
    for g, qs in ansatz_gates(n, params):
        o.apply_gate(g, *qs)
    psi = o.state()
    o.close()
    s = np.arange(1 << n)
    e = 0.0
    for x, z, c in zip(xs, zs, cs):
        sign = 1.0 - 2.0 * (np.bitwise_count(s & z) & 1)
        e += c * np.real(1j ** bin(x & z).count("1") * np.sum(np.conj(psi[s ^ x]) * sign * psi))
    return psi, e


@pytest.mark.parametrize("sizes", [[1], [2, 3], [4, 4, 5, 1, 2], [10, 9, 10, 10, 8], [11], [12, 11, 10, 12, 3, 6]])
@pytest.mark.parametrize("layers,terms", [(0, 3), (1, 1), (2.5, 24), (9, 130)])
def test_energies_and_states(sizes, layers, terms):
    rng = np.random.default_rng(len(sizes) * 100 + terms)
    insts, params = [], []
    for n in sizes:
        xs = [0 if k % 3 == 0 else int(v) for k, v in enumerate(rng.integers(0, 1 << n, terms))]
        zs = [int(v) for v in rng.integers(0, 1 << n, terms)]
        insts.append((n, (xs, zs, [float(v) for v in rng.normal(size=terms)])))
        # a layer is 2 n parameters; half a layer and an odd one left over end inside a layer
        params.append(rng.uniform(-math.pi, math.pi, size=int(2 * n * layers) + (layers == 2.5)))
    b = VqeBatch(insts)
    got = b.evaluate(params)
    for i, ((n, (xs, zs, cs)), p) in enumerate(zip(insts, params)):
        psi, want = exact(n, p, xs, zs, cs)
        assert np.max(np.abs(b.state(i) - psi)) < 1e-12
        assert abs(got[i] - want) < 1e-12 * (1 + sum(abs(c) for c in cs))
    b.close()
