"""GPU tests of the Fock build's implicit quartet spaces: the kernels find the quartets of a
build from the Schwarz bounds and the density maximum on the device."""
import numpy as np
import pytest

import oracle_ffi as O
import unomol_amd
from unomol_amd import api
from unomol_amd.deck import read_deck

pytestmark = pytest.mark.gpu


def _context(tmp_path, kind, n, basis, charge=0):
    path = str(tmp_path / "patin.dat")
    api.generate_deck(path, kind, n, 17, basis, charge, 1e-8, 200)
    b = unomol_amd.Basis(path)
    return read_deck(path), b, unomol_amd.TwoElectronInts(b)


def _density(n, seed, scale):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) * scale
    return np.ascontiguousarray((A + A.T + np.eye(n) * 0.5)[np.tril_indices(n)])


# one function pair; one block per space with idle lanes; several lanes per ket; segments of
# one and of several passes, odd run lengths
@pytest.mark.parametrize("kind,n,basis", [("molecule", 0, "6-31G"), ("water", 1, "6-31G*"), ("water_cluster", 3, "6-31G*"),
                                          ("water_cluster", 11, "6-31G*")])
@pytest.mark.parametrize("scale,tau", [(0.05, 1e-13), (1e-7, 1e-11)])
def test_quartets_within_the_bounds(tmp_path, kind, n, basis, scale, tau):
    """The quartets counted by the launches, FP64 and FP32, against the count from the Schwarz
    bounds and the density maximum: shell pairs (ab) >= (cd) with Qab Qcd 4 max|D| >= tau, FP32
    the ones below the FP32 threshold.  (A product within rounding of a threshold may fall
    either way: one in a million.)"""
    print("[gpu-test] quartet counts %s %d %s" % (kind, n, basis), flush=True)
    deck, b, t = _context(tmp_path, kind, n, basis)
    P = _density(deck["norb"], 3, scale)
    if scale < 1e-6:
        P[:] = np.where(np.abs(P) > 0.1, P * 1e-6, P)
    t.set("schwarz", tau)
    q = np.sort(t.schwarz())[::-1]
    q = q[q > 0.0]
    dmax = np.abs(P).max()
    for prec, thr in ((0, 0.0), (1, 1e-6), (1, 1e30)):
        t.set("precision", prec)
        if prec:
            t.set("fp32_threshold", thr)
        G = np.zeros_like(P)
        t.formGmatrix(P, G)
        cut = lambda lim: sum(int(np.searchsorted(-q[:i + 1], -lim / q[i], side="right")) for i in range(len(q)))  # noqa: E731
        want = cut(tau / (4.0 * dmax))
        want64 = min(want, cut(max(thr, tau / (4.0 * dmax)))) if prec else want
        got, got32 = t.get("last_quartets"), t.get("last_quartets32")
        slack = 1 + want // 1000000
        assert abs(got - want) <= slack, (prec, thr, got, want)
        assert abs(got - got32 - want64) <= slack, (prec, thr, got - got32, want64)


@pytest.mark.parametrize("rows", [0, 1])
@pytest.mark.parametrize("kind,n,basis,charge", [("molecule", 0, "6-31G*", 0), ("molecule", 4, "6-31G*", 1),
                                                 ("water_cluster", 2, "6-31G*", 0)])
def test_small_builds_vs_oracle(tmp_path, kind, n, basis, charge, rows):
    """Builds whose kets are spread over several lanes each, with LDS rows and without, closed
    and open shell, against the oracle's scatter of its own ERIs (1e-11, as the other Fock tests)."""
    print("[gpu-test] small builds %s %d rows %d" % (kind, n, rows), flush=True)
    deck, b, t = _context(tmp_path, kind, n, basis, charge)
    t.set("schwarz", 1e-16)
    t.set("row_merge", rows)
    t.set("row_min_kets", 1)
    val, idx = O.eri_all(deck)
    P = [_density(deck["norb"], 5 + s, 0.05) for s in range(1 + charge)]
    G = [np.zeros_like(p) for p in P]
    t.formGmatrix(*P, *G)
    N = deck["norb"]
    il = np.tril_indices(N)

    def dense(p):
        M = np.zeros((N, N))
        M[il] = p
        return M + np.tril(M, -1).T
    I = np.zeros((N, N, N, N))
    for v, (i, j, k, l) in zip(val, idx):
        for a, c in ((i, j), (j, i)):
            for d, e in ((k, l), (l, k)):
                I[a, c, d, e] = I[d, e, a, c] = v
    D = [dense(p) for p in P]
    J = np.einsum("ijkl,kl->ij", I, 2 * D[0] if len(D) == 1 else D[0] + D[1])
    for g, d in zip(G, D):
        assert np.abs(g - (J - np.einsum("ikjl,kl->ij", I, d))[il]).max() < 1e-11
