"""GPU tests of what the autotuner leaves behind."""
import numpy as np
import pytest

import unomol_amd

pytestmark = pytest.mark.gpu


def _context(tmp_path, waters=6):
    path = str(tmp_path / "w.dat")
    unomol_amd.generate_deck(path, "water_cluster", waters, 3, "6-31G*", 0, 1e-8, 100)
    b = unomol_amd.Basis(path)
    n = b.number_of_orbitals()
    A = 0.05 * np.random.default_rng(1).standard_normal((n, n))
    P = np.ascontiguousarray((A + A.T + np.eye(n))[np.tril_indices(n)])
    return b, unomol_amd.TwoElectronInts(b), P


@pytest.mark.parametrize("mixed", [False, True])
def test_quartet_counts_survive_tuning(tmp_path, mixed):
    """The counts after a tuning build are those of a build of the same density."""
    print("[gpu-test] quartet counts after tuning, mixed %d" % mixed, flush=True)
    b, t, P = _context(tmp_path)
    t.set("row_min_kets", 1)
    t.set("precision", int(mixed))
    t.formGmatrix(P, np.zeros_like(P))
    counts = t.get("last_quartets"), t.get("last_quartets32")
    assert counts[0] > 0 and (counts[1] > 0) == mixed
    assert t.autotune(P, mixed=mixed) > 0.0
    assert (t.get("last_quartets"), t.get("last_quartets32")) == counts
