"""GPU tests of the batched SCF where an exactly degenerate level is half filled on the way: HF, whose
pi pair the first Fock builds leave with one of its two orbitals occupied."""
import numpy as np
import pytest

import unomol_amd
from unomol_amd.deck import parse_deck

pytestmark = pytest.mark.gpu
SEEDS = range(101, 125)
AXES = {"z": (0, 0, 1), "x": (1, 0, 0), "skew": (0.36, -0.48, 0.8)}


def _deck(tmp_path, seed, axis, basis="6-31G"):
    path = str(tmp_path / "hf.dat")
    unomol_amd.generate_deck(path, "molecule", 1, seed, basis, 0, 1e-8, 200)
    with open(path) as f:
        deck = parse_deck(f.read())
    assert list(deck["charge"]) == [9.0, 1.0]
    xyz = np.asarray(deck["xyz"]).reshape(-1, 3)
    deck["xyz"] = np.ascontiguousarray(xyz[0] + np.outer([0.0, np.linalg.norm(xyz[1] - xyz[0])], AXES[axis]))
    return deck


def _densities(decks):
    batch = unomol_amd.Batch(decks)
    out = []
    for _ in range(2):
        e, res = batch.run(cflag=3, eps=1e-8)
        assert all(r.converged for r in res)
        out.append([batch.density(m) for m in range(len(decks))])
    return out


@pytest.mark.parametrize("basis", ["6-31G", "6-31G*"])
@pytest.mark.parametrize("axis", sorted(AXES))
def test_half_filled_pair_repeats(tmp_path, axis, basis):
    """The densities of 24 HF molecules from two runs of one batch, and from batches of a few with a
    water for company (other launches, another order of the Fock sums), agree to 1e-9; the other
    choice of the pair is 2e-7 away.  (Rounding alone leaves less than 1e-11.)"""
    print("[gpu-test] batch, half-filled pi pairs along %s, %s" % (axis, basis), flush=True)
    decks = [_deck(tmp_path, s, axis, basis) for s in SEEDS]
    water = str(tmp_path / "water.dat")
    unomol_amd.generate_deck(water, "water_cluster", 4, 5, "6-31G*", 0, 1e-8, 200)
    runs = _densities(decks)
    parts = [[], []]
    for k in range(0, len(decks), 6):
        for part, got in zip(parts, _densities(decks[k:k + 6] + [water])):
            part.extend(got[:-1])
    for other in runs[1:] + parts:
        for s, a, b in zip(SEEDS, runs[0], other):
            assert np.linalg.norm(a - b) < 1e-9 * np.linalg.norm(a), (s, np.linalg.norm(a - b))


def test_half_filled_pair_along_z_fills_x_first(tmp_path):
    """What exactly equal levels give: the pair in the order of the core Hamiltonian's orbitals, x
    before y, whose density stays the larger by 2e-7 when the energy has converged."""
    decks = [_deck(tmp_path, s, "z") for s in SEEDS]
    print("[gpu-test] batch, half-filled pi pairs, the order", flush=True)
    for s, P in zip(SEEDS, _densities(decks)[0]):
        p = int(np.flatnonzero(np.repeat(decks[0]["sh_l"], (decks[0]["sh_l"] + 1) * (decks[0]["sh_l"] + 2) // 2) == 1)[0])
        assert P[p, p] - P[p + 1, p + 1] > 1e-8, s
