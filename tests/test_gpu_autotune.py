"""GPU tests of what the autotuner leaves behind."""
import numpy as np
import pytest

import unomol_amd
from unomol_amd import _native as N

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


def _launches_by_kind(t, P):
    slots = [np.zeros(432) for _ in range(4)]
    N.check(N.lib().uno_profile(t.ctx, 1, None, None, None, None))
    t.formGmatrix(P, np.zeros_like(P))
    N.check(N.lib().uno_profile(t.ctx, -1, *[N.ptr(s) for s in slots]))
    N.check(N.lib().uno_profile(t.ctx, 0, None, None, None, None))
    return slots[1].reshape(6, 2, 6, 6)[:, 0].sum(axis=(1, 2))


@pytest.mark.parametrize("variant", [1, 2, 3])
def test_forced_layout_goes_before_the_tuned_one(tmp_path, variant):
    """Every launch of the lane kernels (products of up to 162 components) in the forced layout, and
    all of them again as tuned when the knob is back at its default."""
    print("[gpu-test] forced layout %d after tuning" % variant, flush=True)
    b, t, P = _context(tmp_path)
    t.set("row_min_kets", 1)
    assert t.autotune(P) > 0.0
    tuned = _launches_by_kind(t, P)
    t.set("row_variant", variant)
    comps = np.array([1, 3, 9, 6, 18, 36])
    lane = int(((np.multiply.outer(comps, comps) <= 162) & np.tril(np.ones((6, 6), bool))).sum())
    assert _launches_by_kind(t, P)[variant] == lane
    t.set("row_variant", 0)
    assert np.array_equal(_launches_by_kind(t, P), tuned)


def _deck_text(prims):
    """Twelve close atoms (no shell pair is cut) with three s shells each, the first of them a contraction
    of `prims`."""
    first = [(38.36, 0.0238), (5.77, 0.1549), (1.24, 0.4699)][-prims:]
    shells = [(c, s) for c in range(12) for s in (first, [(0.85, 1.0)], [(0.298, 1.0)])]
    text = ["%6d %6d %6d %3d" % (36, 36, 12, 0), "%6d %6d" % (24, 60), " 1e-10", " 0 0", " 2 0 0", " 0 0 0"]
    text += ["2.0 %.6f %.6f %.6f" % (1.0 * (c % 3), 1.05 * (c // 3), 0.02 * c) for c in range(12)]
    for c, s in shells:
        text.append("%3d 0 %d" % (len(s), c))
        text += ["%.10f %.10f" % p for p in s]
    return "\n".join(text) + "\n"


def test_tuning_is_recalled_for_the_same_contraction_only():
    """Two bases of equal functions, shells and pairs whose runs differ in their primitive buckets."""
    print("[gpu-test] tuning recalled by layout", flush=True)
    one, three = unomol_amd.Basis(text=_deck_text(1)), unomol_amd.Basis(text=_deck_text(3))
    t = unomol_amd.TwoElectronInts(three)
    t.set("row_min_kets", 1)
    other = unomol_amd.TwoElectronInts(one)
    assert t.get("pairs") == other.get("pairs") and t.get("pair_runs") != other.get("pair_runs")
    P = np.ascontiguousarray(np.eye(36)[np.tril_indices(36)])
    assert t.autotune(P) > 0.0 and t.get("tuned_launches") == 1
    assert unomol_amd.TwoElectronInts(three).get("tuned_launches") == 1
    assert unomol_amd.TwoElectronInts(one).get("tuned_launches") == 0
