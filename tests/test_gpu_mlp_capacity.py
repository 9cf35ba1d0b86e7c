"""GPU test of the guess network's buffers over calls of growing row counts."""
import numpy as np
import pytest
import torch

import unomol_amd

pytestmark = pytest.mark.gpu


def test_creeping_row_counts_keep_the_buffers():
    """Forward passes of 4200 to 8100 rows, 100 more each time: the device memory in use changes once
    (the first call's), and the last result is that of a fresh network."""
    print("[gpu-test] network buffers over growing row counts", flush=True)
    rng = np.random.default_rng(3)
    X = rng.standard_normal((8100, 128)).astype(np.float32)
    net = unomol_amd.MLP(seed=2)
    free = []
    for n in range(4200, 8101, 100):
        Y = net.forward(X[:n])
        free.append(torch.cuda.mem_get_info()[0])
    assert len(set(free)) == 1, sorted(set(free))
    assert np.array_equal(Y, unomol_amd.MLP(seed=2).forward(X))
