"""Batches that k_mlp_rows and k_mlp_dw take in slices: eight layers of 256 units
hold 1 GiB of activations and gradients for some 87000 rows."""
import ctypes as C

import numpy as np
import pytest

from qcsim_amd._lib import LIB_PATH, check, lib

pytestmark = pytest.mark.gpu
_PF = C.POINTER(C.c_float)


def f(a):
    return a.ctypes.data_as(_PF)


def network(in_dim, hidden, layers):
    h = C.c_void_p()
    check(lib().qcs_mlp_create(in_dim, hidden, layers, 5, C.byref(h)))
    return h, int(lib().qcs_mlp_num_params(h))


def gradients(h, x, t, count):
    g, loss = np.zeros(count, dtype=np.float32), C.c_float()
    check(lib().qcs_mlp_gradients(h, f(x), f(t), len(t), f(g), C.byref(loss)))
    return g, loss.value


# 131072 rows: slices of 86784 and 44288; the network of 300 units runs layer by
# layer, in slices of 69504 and 61568
@pytest.mark.parametrize("hidden", [256, 300])
def test_sums_go_on_from_slice_to_slice(hidden):
    """Rows whose target is the network's own output have no gradient: beside
    them the other half of the batch gives half of what it gives alone, bit for
    bit (a power of two in the mean), before them and after them."""
    h, count = network(3, hidden, 8)
    rng = np.random.default_rng(hidden)
    half = 65536
    x = rng.normal(0, 1, (2 * half, 3)).astype(np.float32)
    y = np.zeros(2 * half, dtype=np.float32)
    check(lib().qcs_mlp_forward(h, f(x), 2 * half, f(y)))
    t = (y + rng.normal(0, 1, y.shape)).astype(np.float32)
    for part in (slice(0, half), slice(half, 2 * half)):
        alone, loss1 = gradients(h, np.ascontiguousarray(x[part]), np.ascontiguousarray(t[part]), count)
        other = y.copy()
        other[part] = t[part]
        both, loss2 = gradients(h, x, other, count)
        assert np.any(alone) and np.array_equal(both, 0.5 * alone)
        assert loss2 == pytest.approx(0.5 * loss1, rel=1e-5)
    lib().qcs_mlp_destroy(h)


def test_training_step_in_slices():
    """One Adam step on the whole data set moves each weight by the learning
    rate against its gradient's sign (the first step's m / sqrt(v) is the sign,
    where the gradient is large beside Adam's epsilon)."""
    h, count = network(3, 256, 8)
    rng = np.random.default_rng(2)
    rows, lr = 100000, 1e-3
    x = rng.normal(0, 1, (rows, 3)).astype(np.float32)
    t = np.sin(x[:, 0]).astype(np.float32)
    before, after, loss = np.zeros(count, np.float32), np.zeros(count, np.float32), np.zeros(1, np.float32)
    check(lib().qcs_mlp_get_params(h, f(before)))
    g, gloss = gradients(h, x, t, count)
    check(lib().qcs_mlp_train(h, f(x), f(t), rows, rows, 1, lr, 3, f(loss)))
    check(lib().qcs_mlp_get_params(h, f(after)))
    lib().qcs_mlp_destroy(h)
    assert loss[0] == pytest.approx(gloss, rel=1e-4)
    big = np.abs(g) > 1e-2 * np.max(np.abs(g))
    assert np.count_nonzero(big) > 100
    # both parameters are rounded to their 24 bits
    np.testing.assert_allclose((after - before)[big], -lr * np.sign(g[big]), atol=1e-2 * lr)


def test_memory_of_a_large_batch():
    """262144 rows through eight layers: the activations and gradients of all
    of them would be 3 GiB; the inputs and per-row outputs are a few MiB."""
    h, count = network(3, 256, 8)
    rng = np.random.default_rng(3)
    x, t = rng.normal(0, 1, (262144, 3)).astype(np.float32), np.zeros(262144, dtype=np.float32)
    hip = C.CDLL(LIB_PATH)  # whose runtime it is

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    before = free()
    gradients(h, x, t, count)
    used = before - free()
    lib().qcs_mlp_destroy(h)
    assert used < 5 << 28
