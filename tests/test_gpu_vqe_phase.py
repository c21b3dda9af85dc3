"""The common factor of a VQE state's Rz rotations."""
import numpy as np
import pytest

from qcsim_amd.vqe import VqeBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rotations", [1, 2, 63, 64, 65, 150])
def test_phase_does_not_lose_with_the_rotations(rotations):
    """Rz rotations alone, of one qubit in |0>: exp(-i sum of the angles / 2).
    Sine and cosine err by an ulp of one at most, the sum of the angles by far
    less: 2^-52, whatever their number."""
    rng = np.random.default_rng(rotations)
    params = []
    for _ in range(200):
        p = np.zeros(2 * rotations)
        p[1::2] = rng.uniform(-np.pi, np.pi, rotations)
        params.append(p)
    batch = VqeBatch([(1, ([0], [1], [1.0]))] * len(params))
    assert np.array_equal(batch.evaluate(params), np.ones(len(params)))
    for i, p in enumerate(params):
        half = np.sum(p[1::2].astype(np.longdouble)) / 2
        psi = batch.state(i)
        assert abs(np.longdouble(psi[0].real) - np.cos(half)) < 2.0**-52
        assert abs(np.longdouble(psi[0].imag) + np.sin(half)) < 2.0**-52
        assert psi[1] == 0
    batch.close()
