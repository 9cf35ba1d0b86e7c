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


def _helium_deck(nfun):
    """A loose, irregular row of helium atoms with three s shells each and the rest on the first."""
    rng = np.random.default_rng(nfun)
    atoms = max(1, nfun // 3)
    extra = nfun - 3 * atoms if nfun >= 3 else 0
    shells = []
    for c in range(atoms):
        prims = [[(38.36, 0.0238), (5.77, 0.1549), (1.24, 0.4699)], [(0.85, 1.0)], [(0.298, 1.0)]]
        shells += [(c, s) for s in prims[: min(3, nfun)]]
    shells += [(0, [(0.11 / (k + 1), 1.0)]) for k in range(extra)]
    text = ["%6d %6d %6d %3d" % (len(shells), len(shells), atoms, 0), "%6d %6d" % (2 * atoms, 60), " 1e-10", " 0 0", " 2 0 0", " 0 0 0"]
    for c in range(atoms):
        x, y, z = 4.0 * c + rng.uniform(-0.3, 0.3), rng.uniform(-1, 1), rng.uniform(-1, 1)
        text.append("2.0 %.12f %.12f %.12f" % (x, y, z))
    for c, s in shells:
        text.append("%3d 0 %d" % (len(s), c))
        text += ["%.10f %.10f" % p for p in s]
    return "\n".join(text) + "\n"


def test_batched_jacobi_sizes():
    """One batch with matrices on both sides of where the eigenvectors leave LDS (98, 99, 100) and
    the matrix does (139, 140, 141), of one and two lanes' worth of pairs (128, 129), and the smallest:
    every energy against the single-molecule SCF's, with the bound of the batch's other test."""
    basis = [unomol_amd.Basis(text=_helium_deck(n)) for n in (1, 2, 3, 98, 99, 100, 128, 129, 139, 140, 141)]
    batch = unomol_amd.Batch([b.deck for b in basis])
    print("[gpu-test] batched jacobi, %d sizes" % len(basis), flush=True)
    e, res = batch.run(maxits=100, eps=1e-10, cflag=3, accel=2)
    for b, eb, r in zip(basis, e, res):
        print("[gpu-test] single scf of %d functions" % b.deck["norb"], flush=True)
        hf = unomol_amd.RestrictedHartreeFock(b, unomol_amd.TwoElectronInts(b))
        es = hf.findEnergy(maxits=100, eps=1e-10, cflag=3, accel=2)
        assert r.converged and hf.result.converged
        assert abs(eb - es) < 1e-8, (b.deck["norb"], eb, es)
