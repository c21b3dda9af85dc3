"""Pauli sums of thousands of terms on hundreds of x masks, as of molecules:
many tile passes, with results fetched many times."""
import numpy as np
import pytest

from qcsim_amd import QubitRegister
from refmath import random_state
from test_gpu_pauli_tiles import reference
from test_pauli_plan import random_terms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,masks,terms", [(6, 40, 700), (12, 300, 2500), (15, 500, 2000)])
def test_many_terms_equal_reference(n, masks, terms, precision):
    rng = np.random.default_rng(n)
    g = QubitRegister(n, precision=precision)
    g.setRegisterStorageFastNoNormalize(random_state(rng, n))
    psi = np.asarray(g.getRegisterStorage()).astype(np.complex128)
    x, z = random_terms(rng, n, masks, terms)
    z = [v | (1 << n - 1) if i % 5 == 0 else v for i, v in enumerate(z)]
    got = g.pauli_expectation(x, z)
    g.close()
    want = np.array([reference(psi, a, b) for a, b in zip(x, z)])
    # sums of 2^n products in FP64 whatever the state's type
    assert np.max(np.abs(got - want)) < 1e-13
