"""GPU tests of the dense eigensolver where its kernels change: the reduction in one block up to 192 and
by column launches above, one eigenvector or several per block of the inverse iteration, chunks of 16
rows; and the batched Jacobi's three placements of its matrices."""
import numpy as np
import pytest

import unomol_amd

pytestmark = pytest.mark.gpu


def _matrix(n, kind):
    rng = np.random.default_rng(n)
    if kind == "random":
        A = rng.standard_normal((n, n))
    elif kind == "degenerate":
        q, _ = np.linalg.qr(rng.standard_normal((n, n)))
        ev = rng.uniform(-20, 5, n)
        ev[: n // 2] = np.repeat(ev[: (n // 2 + 2) // 3], 3)[: n // 2]
        A = (q * ev) @ q.T
    elif kind == "split":   # decoupled blocks: zero reflectors and off-diagonals
        A = np.zeros((n, n))
        for lo in range(0, n, 7):
            hi = min(n, lo + 7)
            A[lo:hi, lo:hi] = rng.standard_normal((hi - lo, hi - lo))
    else:
        A = np.diag(np.arange(n, dtype=float))
    return A + A.T


@pytest.mark.parametrize("n", [3, 4, 16, 17, 33, 65, 191, 192, 193, 257, 321, 1216])
@pytest.mark.parametrize("kind", ["random", "degenerate", "split", "diagonal"])
def test_eigensolver_edges(n, kind):
    """Against numpy, with the bounds of the solver's other test."""
    print("[gpu-test] eigh %s n=%d" % (kind, n), flush=True)
    A = _matrix(n, kind)
    i, j = np.tril_indices(n)
    z, e = np.zeros(n * n), np.zeros(n)
    unomol_amd.SymmPack.rsp(n, np.ascontiguousarray(A[i, j]), z, e)
    Z = z.reshape(n, n)
    ref = np.linalg.eigvalsh(A)
    scale = max(1.0, np.abs(ref).max())
    tol = max(1, n / 10)
    assert np.abs(e - ref).max() < 1e-13 * scale * tol
    assert np.all(np.diff(e) >= 0)
    assert np.abs(A @ Z - Z * e).max() < 1e-12 * scale * tol
    assert np.abs(Z.T @ Z - np.eye(n)).max() < 1e-12 * tol
