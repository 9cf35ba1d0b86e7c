"""GPU tests of which shell pairs a context keeps, and of the quartet spaces made of them, against a
plain loop over primitive pairs."""
import numpy as np
import pytest

import unomol_amd

pytestmark = pytest.mark.gpu


def _deck(seed):
    """Fragments 2 to 30 bohr apart: atoms with a tight contraction, a mixed one and a diffuse
    primitive each, some with p and d shells, so that pairs end at every distance."""
    rng = np.random.default_rng(seed)
    kinds = [(0, [(180.0, 0.02), (27.0, 0.15), (6.1, 0.5), (1.7, 0.45)]), (0, [(2.9, 0.4), (0.31, 0.7)]), (0, [(0.052, 1.0)]),
             (1, [(7.8, 0.1), (1.6, 0.4), (0.41, 0.6)]), (1, [(0.09, 1.0)]), (2, [(0.8, 1.0)])]
    xyz = np.cumsum(np.concatenate([[0.0], rng.uniform(2.0, 6.0, 4), [30.0], rng.uniform(2.0, 4.0, 3), [11.0]]))
    shells = [(c, l, prims) for c in range(len(xyz)) for l, prims in kinds if l == 0 or (c + l) % 3 == 0]
    nfun = sum((l + 1) * (l + 2) // 2 for _, l, _ in shells)
    text = ["%6d %6d %6d %3d" % (len(shells), nfun, len(xyz), 2), "%6d %6d" % (2 * len(xyz), 60), " 1e-10", " 0 0", " 2 0 0", " 0 0 0"]
    text += ["2.0 %.12f %.12f %.12f" % (x, rng.uniform(-1, 1), rng.uniform(-1, 1)) for x in xyz]
    for c, l, prims in shells:
        text.append("%3d %d %d" % (len(prims), l, c))
        text += ["%.10f %.10f" % p for p in prims]
    return "\n".join(text) + "\n"


def _kept(deck, cut):
    """Primitive pairs of every shell pair whose bare prefactor with the most diffuse ket,
    2 pi^(5/2) exp(-ab/p R^2) / (p q sqrt(p + q)), reaches the cut (same shell: a triangle)."""
    low = 2.0 * deck["alpha"].min()
    ex = [deck["alpha"][o:o + k] for o, k in zip(deck["sh_poff"], deck["sh_npr"])]
    xyz = np.asarray(deck["xyz"]).reshape(-1, 3)[deck["sh_cen"]]
    out = {}
    for a in range(len(ex)):
        for b in range(a + 1):
            p = ex[a][:, None] + ex[b][None]
            s = np.exp(-ex[a][:, None] * ex[b][None] / p * ((xyz[a] - xyz[b]) ** 2).sum())
            keep = 2 * np.pi ** 2.5 * s / (p * low * np.sqrt(p + low)) >= cut
            if a == b:
                keep = np.tril(keep)
            if keep.any():
                hi, lo = max(deck["sh_l"][a], deck["sh_l"][b]), min(deck["sh_l"][a], deck["sh_l"][b])
                out[a, b] = (int(hi), int(lo), int(keep.sum()))
    return out


@pytest.mark.parametrize("cut", [1e-12, 1e-20, 1e-5, 0.0])
@pytest.mark.parametrize("seed", [1, 2])
def test_pairs_against_a_primitive_loop(cut, seed):
    """The number of pairs and of their runs (a class and a bucket of primitive counts each), and one
    space in the launches' tables for every two runs, an equal pair of them included."""
    print("[gpu-test] shell pairs, cut %g" % cut, flush=True)
    b = unomol_amd.Basis(text=_deck(seed))
    t = unomol_amd.TwoElectronInts(b)
    t.set("prim_cut", cut)
    t.recalculate(b)
    want = _kept(b.deck, cut)
    ns = b.deck["nshell"]
    if cut > 0.0:
        assert ns < len(want) < ns * (ns + 1) // 2   # the cut falls between the pairs
    assert int(t.get("pairs")) == len(want)
    runs = {(h, l, int(np.searchsorted([1, 3, 6, 9, 18], k))) for h, l, k in want.values()}
    assert int(t.get("pair_runs")) == len(runs)
    assert int(t.get("quartet_launches")) == len(runs) * (len(runs) + 1) // 2
    q = t.schwarz()
    for a in range(ns):
        for c in range(a + 1):
            assert (a, c) in want or q[a * (a + 1) // 2 + c] == 0.0


@pytest.mark.parametrize("molecules", [1, 3])
def test_spaces_of_a_batch_are_built_once(tmp_path, molecules):
    """Two runs of a batch capture its build twice, over the spaces made with the batch."""
    path = str(tmp_path / "w.dat")
    unomol_amd.generate_deck(path, "water", 1, 3, "6-31G", 0, 1e-8, 100)
    batch = unomol_amd.Batch([path] * molecules)
    assert batch.get("space_builds") == 1
    for _ in range(2):
        _, res = batch.run(maxits=100, eps=1e-8, cflag=3)
        assert batch.get("graph_builds") == 1 and batch.get("graph_replays") == max(r.iterations for r in res)
        assert batch.get("space_builds") == 1
    # one launch per class pair: ss, ps, pp against each other
    assert batch.get("launches_per_build") == 6
