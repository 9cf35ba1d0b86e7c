"""GPU tests of every LDS layout of the Fock kernels, each forced and seen to run."""
import numpy as np
import pytest

import oracle_ffi as O
import unomol_amd
from unomol_amd import _native as N
from unomol_amd.deck import read_deck

pytestmark = pytest.mark.gpu


def _launches_by_kind(t, build):
    slots = [np.zeros(432) for _ in range(4)]
    N.check(N.lib().uno_profile(t.ctx, 1, None, None, None, None))
    build()
    N.check(N.lib().uno_profile(t.ctx, -1, *[N.ptr(s) for s in slots]))
    N.check(N.lib().uno_profile(t.ctx, 0, None, None, None, None))
    return slots[1].reshape(6, 2, 6, 6)[:, 0]


@pytest.mark.parametrize("charge", [0, 1])
@pytest.mark.parametrize("variant", [1, 2, 3])
@pytest.mark.parametrize("dens", [-1, 0, 1])
def test_forced_layouts_vs_oracle(tmp_path, variant, dens, charge):
    """G of an H2O in 6-31G*, closed shell and cation, against the oracle's scatter of its own ERIs
    (1e-11, as the other Fock tests); every class of the lane kernels took the forced layout."""
    print("[gpu-test] fock layout %d, density rows %d, charge %d" % (variant, dens, charge), flush=True)
    path = str(tmp_path / "patin.dat")
    unomol_amd.generate_deck(path, "water", 1, 7, "6-31G*", charge, 1e-8, 100)
    deck = read_deck(path)
    b = unomol_amd.Basis(path)
    t = unomol_amd.TwoElectronInts(b)
    for key, v in (("schwarz", 1e-16), ("row_min_kets", 1), ("row_variant", variant), ("row_density_lds", dens)):
        t.set(key, v)
    n = deck["norb"]
    rng = np.random.default_rng(variant)
    il = np.tril_indices(n)
    D = [A + A.T for A in (0.1 * rng.standard_normal((n, n)) for _ in range(1 + charge))]
    P = [np.ascontiguousarray(d[il]) for d in D]
    G = [np.zeros_like(p) for p in P]
    launches = _launches_by_kind(t, lambda: t.formGmatrix(*P, *G))
    comps = np.array([1, 3, 9, 6, 18, 36])
    lane = (np.multiply.outer(comps, comps) <= 162) & np.tril(np.ones((6, 6), bool))
    wave = ~lane & np.tril(np.ones((6, 6), bool))
    assert np.all(launches[variant][lane] == 1) and np.all(launches[0][wave] == 1)
    assert launches.sum() == 21
    I = np.zeros((n, n, n, n))
    for v, (i, j, k, l) in zip(*O.eri_all(deck)):
        for a, c in ((i, j), (j, i)):
            for d, e in ((k, l), (l, k)):
                I[a, c, d, e] = I[d, e, a, c] = v
    J = np.einsum("ijkl,kl->ij", I, 2 * D[0] if charge == 0 else D[0] + D[1])
    for g, d in zip(G, D):
        assert np.abs(g - (J - np.einsum("ikjl,kl->ij", I, d))[il]).max() < 1e-11
