"""Measurements whose outcome stays on the device until the collapse: states of
one chunk (1..11 qubits, one launch), of a few (12, 13) and with the large
sum (22), single and ranged qubits, uniforms at the ends, and samplings
around what the register's scratch holds (4096 shots)."""
import numpy as np
import pytest

from qcsim_amd import QubitRegister
from refmath import cdf_first, random_state

pytestmark = pytest.mark.gpu


def register(n, precision, seed):
    g = QubitRegister(n, precision=precision)
    g.setRegisterStorageFastNoNormalize(random_state(np.random.default_rng(seed), n))
    return g, np.asarray(g.getRegisterStorage()).astype(np.complex128)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 5, 8, 11, 12, 13, 22])
def test_measure_and_collapse(n, precision):
    rng = np.random.default_rng(n)
    for first, second in {(0, 0), (n - 1, n - 1), (0, n - 1), (n // 2, min(n - 1, n // 2 + 2))}:
        # the ends, but for probability 1, which lies within the rounding of the sum
        for u in (1e-12, float(rng.random()), float(rng.random()), 1.0 - 2.0**-53):
            g, psi = register(n, precision, 7 * n)
            st = cdf_first(psi, 1.0 - u, 0)
            mask = ((2 << second) - 1) & ~((1 << first) - 1)
            assert g.Measure(first, second, u=u) == (st & mask) >> first
            keep = (np.arange(1 << n) & mask) == (st & mask)
            want = np.where(keep, psi, 0) / np.sqrt(np.sum(np.abs(psi[keep]) ** 2))
            # one rounding of each part of a stored amplitude
            assert np.max(np.abs(g.getRegisterStorage() - want)) < (1e-14 if precision == "c128" else 1.2e-7)
            g.close()
    g, psi = register(n, precision, 7 * n)
    u = float(rng.random())
    st = cdf_first(psi, 1.0 - u, (1 << n) - 1)
    assert g.MeasureNoCollapse(u=u) == st and g.MeasureAll(u=u) == st
    assert np.array_equal(g.getRegisterStorage(), np.arange(1 << n) == st)
    g.close()


@pytest.mark.parametrize("n", [3, 11, 12, 16])
@pytest.mark.parametrize("shots", [1, 2, 4096, 4097, 70000])
def test_sampling(n, shots):
    g, psi = register(n, "c128", n)
    u = np.random.default_rng(shots).random(shots)
    u[: shots // 7] *= 1e-16  # beyond the truncation of the CDF
    c = np.cumsum(psi.real * psi.real + psi.imag * psi.imag)
    got = g.sample(u)
    if shots == 1:
        want = np.array([cdf_first(psi, 1.0 - u[0], 0)])
        near = np.zeros(1, bool)
    else:
        top = int(np.searchsorted(c, 1.0 - np.finfo(float).eps, side="right"))
        length = min(top + 1, 1 << n)
        want = np.searchsorted(c[:length], 1.0 - u, side="left")
        # the prefix sums of chunks differ from the sequential ones by rounding
        i = np.minimum(np.searchsorted(c, 1.0 - u), (1 << n) - 1)
        near = np.minimum(np.abs(c[i] - (1.0 - u)), np.abs(c[np.maximum(i - 1, 0)] - (1.0 - u))) < 1e-14
    assert np.array_equal(got[~near], want[~near])
    g.close()
