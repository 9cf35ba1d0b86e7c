"""GPU tests of the kernels that run once per geometry: Schwarz bounds whose lanes share a pair's
primitives, and one-electron integrals whose lanes share primitives and nuclei."""
import numpy as np
import pytest

import unomol_amd

pytestmark = pytest.mark.gpu


def _deck(tmp_path, waters, basis):
    path = str(tmp_path / "deck.dat")
    unomol_amd.generate_deck(path, "water_cluster", waters, 3, basis, 0, 1e-8, 50)
    return path


# every pair class and 1 to 36 primitive pairs (one lane's share empty, ragged, several rounds)
@pytest.mark.parametrize("waters,basis", [(1, "6-31G"), (1, "6-31G*"), (2, "6-31G*")])
def test_schwarz_is_the_largest_diagonal(tmp_path, waters, basis):
    """Every bound against the (ij|ij) of the explicit integrals.  Both sum at most 1296 products
    in double: 1296 x 2^-53 x a few roundings each is below 1e-12 of the summed magnitudes, which
    stay below 10."""
    print("[gpu-test] schwarz bounds %d %s" % (waters, basis), flush=True)
    b = unomol_amd.Basis(_deck(tmp_path, waters, basis))
    t = unomol_amd.TwoElectronInts(b)
    t.set("prim_cut", 0.0)
    t.recalculate(b)
    val, f = t.eri_emit()
    d = b.deck
    nfun = (np.asarray(d["sh_l"]) + 1) * (np.asarray(d["sh_l"]) + 2) // 2
    shell = np.repeat(np.arange(len(nfun)), nfun)
    diag = (f[:, 0] == f[:, 2]) & (f[:, 1] == f[:, 3])
    a, c = shell[f[diag, 0]], shell[f[diag, 1]]
    ref = np.zeros(len(nfun) * (len(nfun) + 1) // 2)
    np.maximum.at(ref, np.maximum(a, c) * (np.maximum(a, c) + 1) // 2 + np.minimum(a, c), np.abs(val[diag]))
    q = t.schwarz()
    assert np.abs(q * q - ref).max() < 1e-11


# fewer nuclei than lanes; one and several primitive pairs at a time
@pytest.mark.parametrize("waters", [1, 7, 8, 23])
def test_oneint_lane_shares(tmp_path, waters):
    """Against the host's integrals, with the bounds of the device integrals' other test scaled by
    the number of nuclei, whose terms are what is summed in another order."""
    print("[gpu-test] one-electron integrals, %d waters" % waters, flush=True)
    b = unomol_amd.Basis(_deck(tmp_path, waters, "6-31G*"))
    t = unomol_amd.TwoElectronInts(b)
    for dev, host in zip(t.oneint(), unomol_amd.oneint(b.deck)):
        assert np.abs(dev - host).max() < 1e-13 * max(1.0, np.abs(host).max()) * waters
