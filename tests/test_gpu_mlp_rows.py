"""The surrogate's matrix kernels at the edges of their tiles: inputs and
widths around the paddings (32, 64, 128, 256), networks one unit too wide for
them (layer by layer instead), batches around the row tiles and the gradient
slabs. Forward outputs equal the FP32 sums in ascending order bit for bit;
loss and gradients are held to the oracle at the bounds of test_gpu_mlp.py."""
import ctypes as C

import numpy as np
import pytest

from oracle.mlp_ref import bf16_round, loss_and_grad, unpack
from qcsim_amd._lib import check, lib

pytestmark = pytest.mark.gpu
_PF = C.POINTER(C.c_float)


def chain(a, w):
    """a @ w with one FP32 FMA per term, k ascending: BF16 products and their
    sums with an FP32 value are exact in FP64 (up to 53 bits apart), so one
    rounding per term remains."""
    acc = np.zeros((a.shape[0], w.shape[1]), dtype=np.float32)
    for k in range(a.shape[1]):
        acc = (acc.astype(np.float64) + np.outer(a[:, k], w[k])).astype(np.float32)
    return acc


def forward_f32(params, dims, x):
    a = bf16_round(x)
    layers = unpack(params, dims)
    for W, b in layers[:-1]:
        z = chain(a, bf16_round(W)) + b.astype(np.float32)
        a = bf16_round(np.maximum(z, np.float32(0)))
    W, b = layers[-1]
    return (chain(a, bf16_round(W)) + b.astype(np.float32))[:, 0]


@pytest.mark.parametrize(
    "in_dim,hidden,layers,batch",
    [(1, 1, 1, 1), (17, 256, 3, 17), (32, 64, 2, 16), (33, 65, 2, 255), (256, 128, 1, 257), (31, 129, 8, 33),
     (11, 200, 2, 8193), (256, 257, 2, 40), (257, 16, 2, 300)],
)
def test_edges_match_the_ordered_sums_and_the_oracle(in_dim, hidden, layers, batch):
    rng = np.random.default_rng(in_dim * 1000 + hidden)
    h = C.c_void_p()
    check(lib().qcs_mlp_create(in_dim, hidden, layers, 5, C.byref(h)))
    dims = [in_dim] + [hidden] * layers + [1]
    p = np.zeros(lib().qcs_mlp_num_params(h), dtype=np.float32)
    check(lib().qcs_mlp_get_params(h, p.ctypes.data_as(_PF)))
    p = p + rng.normal(0, 0.05, p.shape).astype(np.float32)
    check(lib().qcs_mlp_set_params(h, p.ctypes.data_as(_PF)))
    x = rng.normal(0, 1, (batch, in_dim)).astype(np.float32)
    t = rng.normal(0, 1, batch).astype(np.float32)
    y = np.zeros(batch, dtype=np.float32)
    for _ in range(2):
        check(lib().qcs_mlp_forward(h, x.ctypes.data_as(_PF), batch, y.ctypes.data_as(_PF)))
        assert np.array_equal(y, forward_f32(p, dims, x))
    g = np.zeros(p.shape[0], dtype=np.float32)
    loss = C.c_float()
    check(lib().qcs_mlp_gradients(h, x.ctypes.data_as(_PF), t.ctypes.data_as(_PF), batch, g.ctypes.data_as(_PF),
                                  C.byref(loss)))
    l_ref, g_ref = loss_and_grad(p.astype(np.float64), dims, x, t)
    assert abs(loss.value - l_ref) < 2e-3 * (1 + l_ref)
    assert np.linalg.norm(g - g_ref) < 1e-2 * np.linalg.norm(g_ref)
    lib().qcs_mlp_destroy(h)
