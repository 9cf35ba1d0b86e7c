"""GPU tests of the dense eigensolver where its kernels' shared memory passes 64 KB and where it ends."""
import numpy as np
import pytest
import torch

import unomol_amd
from unomol_amd._native import UnoError

pytestmark = pytest.mark.gpu
LARGEST = 6752   # three vectors of it are a block's 160 KB


def _solve(n):
    A = torch.randn(n, n, dtype=torch.float64, generator=torch.Generator().manual_seed(n))
    A = (A + A.T) / np.sqrt(n)
    i, j = torch.tril_indices(n, n)
    z, e = np.zeros(n * n), np.zeros(n)
    unomol_amd.SymmPack.rsp(n, np.ascontiguousarray(A[i, j].numpy()), z, e)
    return A, torch.from_numpy(z).reshape(n, n), torch.from_numpy(e)


# the bisection's arrays above 64 KB (n > 4096); the largest size
@pytest.mark.parametrize("n", [4097, LARGEST])
def test_large_matrices(n):
    """Residual and orthogonality with the bounds of the solver's other tests."""
    print("[gpu-test] eigh n=%d" % n, flush=True)
    A, Z, e = (x.cuda() for x in _solve(n))
    scale, tol = max(1.0, float(e.abs().max())), n / 10
    assert bool((e[1:] >= e[:-1]).all())
    assert float((A @ Z - Z * e).abs().max()) < 1e-12 * scale * tol
    assert float((Z.T @ Z - torch.eye(n, dtype=torch.float64, device="cuda")).abs().max()) < 1e-12 * tol


def test_beyond_the_largest_is_an_error():
    n = LARGEST + 1
    z, e = np.zeros(n * n), np.zeros(n)
    with pytest.raises(UnoError, match="largest size"):
        unomol_amd.SymmPack.rsp(n, np.zeros(n * (n + 1) // 2), z, e)
