"""The kernel that closes a turn (moments of every bunch, wake of its bins)
at the edges of its split: segment counts around a wave's 64 lanes and its
four-segment steps, bin counts around the 64 bins of a block and the eight
parts of its sum.  Moments against numpy on the downloaded coordinates
(sums of n values: within 1e-11 of the rms size), wake kicks against numpy's
sum over the bins with the oracle's lag table (at most 1024 terms: within
1e-12 of the largest kick)."""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.tracker import COORDS, Tracker

import oracle as O

pytestmark = pytest.mark.gpu

BBR = configs.BASE["bbr"]
SZ = configs.BASE["sig"][2]


def bunch(n, seed):
    ring, secs, _ = configs.lattice()
    tr = Tracker(ring, secs)
    q, ne = configs.bunch_scalars([n], ring)
    tr.set_bunches([n], q, ne)
    tr.upload(configs.gaussian_bunch(n, seed))
    return ring, tr, q[0]


@pytest.mark.parametrize("nseg", [1, 2, 63, 64, 65, 255, 256, 257, 513])
def test_moments_of_any_segment_count(nseg):
    n = 256 * (nseg - 1) + 17
    ring, tr, _ = bunch(n, 3)
    tr.set_wake(50, 1, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
    tr.set_layout(nseg, 256)
    tr.set_history(2)
    print(f"moments of {nseg} segments", flush=True)
    for t in range(2):
        tr.turn(t)
    m = tr.moments()[0]
    h = tr.history(1, 1)[0]
    d = tr.download()
    v = [d[c] for c in COORDS]
    sig = [np.std(x) for x in v]
    assert m["n_alive"] == n
    for i in range(6):
        assert abs(m["mean"][i] - np.mean(v[i])) <= 1e-11 * sig[i], i
    pairs = ((0, 0), (0, 1), (1, 1), (2, 2), (2, 3), (3, 3), (4, 4), (4, 5), (5, 5))
    for k, (i, j) in enumerate(pairs):
        exp = np.mean((v[i] - np.mean(v[i])) * (v[j] - np.mean(v[j])))
        assert abs(m["c2"][k] - exp) <= 1e-11 * sig[i] * sig[j], k
    assert m["zmin"] == np.min(v[4]) and m["zmax"] == np.max(v[4])
    assert np.array_equal(h["mean"], m["mean"]) and np.array_equal(h["c2"], m["c2"])
    tr.close()


@pytest.mark.parametrize("nbins", [1, 2, 7, 8, 9, 63, 64, 65, 129, 1024])
def test_wake_of_any_bin_count(nbins):
    n = 5000
    ring, tr, q = bunch(n, 4)
    print(f"wake of {nbins} bins", flush=True)
    tr.set_wake(nbins, 1, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
    tr.turn(0)
    counts, edges, kick = tr.wake_state()
    z = tr.download()["z"]
    k = np.trunc((z - edges[0, 0]) / edges[0, 1]).astype(int)
    assert np.array_equal(counts[0], np.bincount(k[(k >= 0) & (k < nbins)], minlength=nbins))
    rs, qq, om = (np.array(BBR[c], float) for c in ("rs", "q", "fr"))
    table = np.zeros(2 * nbins - 1)
    O.lib().orc_wake_table(nbins, edges[0, 1] / configs.C_LIGHT, len(rs), O.p(rs), O.p(qq), O.p(om * 2 * np.pi),
                           O.p(table))
    i = np.arange(nbins)
    exp = table[i[:, None] - i[None, :] + nbins - 1] @ counts[0] * (-configs.E_CHARGE * q / ring.energy)
    assert np.max(np.abs(exp)) > 0
    assert np.max(np.abs(kick[0] - exp)) <= 1e-12 * np.max(np.abs(exp))
    tr.close()
