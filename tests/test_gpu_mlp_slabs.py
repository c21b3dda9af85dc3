"""The weight gradients' slabs (192 rows, four in LDS): batches around one and
several slabs and fewer rows than a group of 32, widths around the 32 x 32
tiles and the column of ones. The gradient of the last bias is a sum over the
rows alone, so a lost, repeated or stale row shows; the others are held to the
oracle."""
import ctypes as C

import numpy as np
import pytest

from oracle.mlp_ref import loss_and_grad
from qcsim_amd._lib import check, lib

pytestmark = pytest.mark.gpu
_PF = C.POINTER(C.c_float)


@pytest.mark.parametrize("in_dim,hidden", [(17, 64), (31, 32), (32, 96), (63, 256)])
@pytest.mark.parametrize("batch", [5, 32, 191, 192, 193, 383, 385, 576, 769, 961])
def test_gradients_at_slab_edges(in_dim, hidden, batch):
    rng = np.random.default_rng(in_dim + batch)
    h = C.c_void_p()
    check(lib().qcs_mlp_create(in_dim, hidden, 2, 5, C.byref(h)))
    dims = [in_dim, hidden, hidden, 1]
    n = lib().qcs_mlp_num_params(h)
    p, g = np.zeros(n, dtype=np.float32), np.zeros(n, dtype=np.float32)
    check(lib().qcs_mlp_get_params(h, p.ctypes.data_as(_PF)))
    loss = C.c_float()
    for rows in (961, batch):  # a larger batch first: its rows lie behind the smaller one's
        x = rng.normal(0, 1, (rows, in_dim)).astype(np.float32)
        t = rng.normal(0, 1, rows).astype(np.float32)
        check(lib().qcs_mlp_gradients(h, x.ctypes.data_as(_PF), t.ctypes.data_as(_PF), rows, g.ctypes.data_as(_PF),
                                      C.byref(loss)))
    y = np.zeros(batch, dtype=np.float32)
    check(lib().qcs_mlp_forward(h, x.ctypes.data_as(_PF), batch, y.ctypes.data_as(_PF)))
    check(lib().qcs_mlp_destroy(h))
    d = 2.0 * (y.astype(np.float64) - t) / batch
    # one FP32 rounding a row, and those of the rows themselves
    assert abs(g[-1] - d.sum()) < (batch + 4) * 2.0**-24 * np.abs(d).sum()
    _, ref = loss_and_grad(p, dims, x, t)
    assert np.linalg.norm(g - ref) < 1e-2 * np.linalg.norm(ref)
