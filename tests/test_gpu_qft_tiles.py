"""The QFT's passes above the lowest twelve qubits at each split of their
targets: none to four and ten or eleven (registers), five to nine in one tile
pass, more in two, ranges that begin and end inside the register, both
directions, with and without the swaps, against numpy's FFT."""
import numpy as np
import pytest

from qcsim_amd import QubitRegister
from refmath import qft_closed, random_state

pytestmark = pytest.mark.gpu


def reversed_bits(v, n, sq, eq):
    """The state with the qubits of the range in the opposite order."""
    m = eq - sq + 1
    axes = list(range(n))
    top = n - 1 - eq
    axes[top : top + m] = axes[top : top + m][::-1]
    return v.reshape([2] * n).transpose(axes).reshape(-1)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,sq,eq", [(13, 0, 12), (16, 0, 15), (17, 0, 16), (18, 2, 17), (19, 0, 17), (20, 0, 19),
                                     (21, 0, 20), (22, 0, 21), (22, 12, 21), (22, 14, 20), (23, 0, 22), (24, 0, 23),
                                     (24, 5, 23)])
def test_qft_equals_fft(n, sq, eq, precision):
    rng = np.random.default_rng(n * 100 + sq)
    g = QubitRegister(n, precision=precision)
    g.setRegisterStorageFastNoNormalize(random_state(rng, n))
    psi = np.asarray(g.getRegisterStorage()).astype(np.complex128)
    # a target costs a phase and a butterfly, four roundings of an amplitude
    tol = 4 * n * (2.0**-53 if precision == "c128" else 2.0**-24) * 4
    for inverse in (False, True):
        for swap in (True, False):
            g.setRegisterStorageFastNoNormalize(psi.copy())
            g.qft(sq, eq, do_swap=swap, inverse=inverse)
            src = psi if swap or not inverse else reversed_bits(psi, n, sq, eq)
            want = qft_closed(src, n, sq, eq, inverse=inverse)
            if not swap and not inverse:
                want = reversed_bits(want, n, sq, eq)
            assert np.linalg.norm(g.getRegisterStorage() - want) < tol, (inverse, swap)
    g.close()
