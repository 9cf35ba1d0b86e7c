"""GPU tests of the guess network's row handling: padded rows, and the weight gradient's split
of a batch into row chunks."""
import os
import sys

import numpy as np
import pytest

import unomol_amd
from unomol_amd._native import UnoError

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as MO  # noqa: E402

pytestmark = pytest.mark.gpu


# one row; a tile less and more one row; one chunk's and the largest chunk count's edges; chunks of
# 128 rows with a short last one
@pytest.mark.parametrize("n", [1, 63, 65, 2048, 2049, 4161])
def test_gradient_over_row_chunks(n):
    """Loss and gradient against the numpy oracle with the same BF16 roundings, with the
    tolerance of the network's other gradient test, and the gradient of a repeated call bitwise."""
    print("[gpu-test] mlp gradient, %d rows" % n, flush=True)
    rng = np.random.default_rng(n)
    net = unomol_amd.MLP(64, 128, 2, 64, seed=3)
    X = rng.standard_normal((n, 64)).astype(np.float32)
    T = rng.standard_normal((n, 64)).astype(np.float32)
    M = (rng.random((n, 64)) < 0.7).astype(np.float32)
    M[0, 0] = 1.0
    loss, g = net.loss_grad(X, T, M)
    lref, gref = MO.loss_grad(net.get_params(), net.dims, X, T, M)
    assert abs(loss - lref) < 1e-3 * abs(lref)
    assert np.linalg.norm(g - gref) < 1e-2 * np.linalg.norm(gref)
    loss2, g2 = net.loss_grad(X, T, M)
    assert loss2 == loss and np.array_equal(g2, g)


def test_empty_mask_is_an_error():
    net = unomol_amd.MLP(64, 64, 1, 64, seed=1)
    Z = np.zeros((5, 64), dtype=np.float32)
    with pytest.raises(UnoError):
        net.loss_grad(Z, Z, Z)
