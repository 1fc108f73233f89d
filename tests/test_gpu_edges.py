"""The reference's bin edges (the survivors' z range after the turn, widened by
two rms of z after the section map, which leaves z alone in this ring) with
the bins and the lag table formed in the turn's closing kernel: bunches around
the share of a binning block, segment counts around the fold's four, bin
counts around a wave.  Edges against numpy (rms from sums of n values: 1e-11
of the width), counts against numpy on the kernel's own edges (whole numbers,
but for values within 1e-9 of an edge), kicks against numpy's sum with the
oracle's table (at most 129 terms: 1e-12 of the largest).

And the stage sets compiled for one kind of turn, over the wakes, the radiation
models and the long-range wake.  A flush between turns only moves the deferred
kick to a pass of its own: the same coordinates, loss codes and bins.  They equal
the general set's, reached with a second RF term of voltage zero, which adds
exact zeros; with radiation, whose stage rounds once where it can fuse, up to
those roundings.
"""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.tracker import COORDS, Tracker

import oracle as O

pytestmark = pytest.mark.gpu

BBR = configs.BASE["bbr"]
SZ = configs.BASE["sig"][2]


@pytest.mark.parametrize("nbins,counts,layout", [
    (1, [3000], None), (8, [4095, 4096, 4097], None), (64, [100], (1, 0)), (65, [530_000, 7000], None),
    (129, [20_000], (3, 0)), (64, [9000, 255, 70_001], (5, 0)), (50, [1025], (257, 4))])
def test_reference_edges(nbins, counts, layout):
    ring, secs, _ = configs.lattice()
    nb = len(counts)
    q, ne = configs.bunch_scalars(counts, ring)
    tr = Tracker(ring, secs)
    tr.set_bunches(counts, q, ne, configs.train_gaps(nb, 1, ring.harmonic) if nb > 1 else None)
    tr.upload(configs.gaussian_bunch(int(np.sum(counts)), 6))
    tr.set_wake(nbins, 0, 0.0, 0.0, BBR["rs"], BBR["q"], BBR["fr"])
    if layout:
        tr.set_layout(*layout)
    print(f"edges of {counts} macroparticles, {nbins} bins", flush=True)
    tr.turn(0)
    z_map = tr.download()["z"]
    tr.turn(1)
    cnt, edges, kick = tr.wake_state()
    mom = tr.moments()
    off = np.concatenate([[0], np.cumsum(counts)])
    z_all = tr.download()["z"]
    rs, qq, om = (np.array(BBR[c], float) for c in ("rs", "q", "fr"))
    for b in range(nb):
        z = z_all[off[b]:off[b + 1]]
        assert mom[b]["zmin"] == z.min() and mom[b]["zmax"] == z.max()
        sig = np.std(z_map[off[b]:off[b + 1]])
        lo, hi = z.min() - 1e-6 - 2 * sig, z.max() + 1e-6 + 2 * sig
        assert abs(edges[b, 0] - lo) <= 1e-11 * (hi - lo)
        assert abs(edges[b, 1] * nbins - (hi - lo)) <= 1e-11 * (hi - lo)
        f = (z - edges[b, 0]) / edges[b, 1]
        near = int(np.sum(np.abs(f - np.rint(f)) < 1e-9))
        exp = np.bincount(np.trunc(f).astype(int), minlength=nbins)[:nbins]
        assert cnt[b].sum() == len(z) and np.abs(cnt[b].astype(int) - exp).sum() <= 2 * near
        table = np.zeros(2 * nbins - 1)
        O.lib().orc_wake_table(nbins, edges[b, 1] / configs.C_LIGHT, len(rs), O.p(rs), O.p(qq),
                               O.p(om * 2 * np.pi), O.p(table))
        i = np.arange(nbins)
        want = table[i[:, None] - i[None, :] + nbins - 1] @ cnt[b] * (-configs.E_CHARGE * q[b] / ring.energy)
        assert np.max(np.abs(kick[b] - want)) <= 1e-12 * np.max(np.abs(want))
    tr.close()


@pytest.mark.parametrize("wake", [None, 0, 1])
@pytest.mark.parametrize("noise", [None, 1, 2])
@pytest.mark.parametrize("lrw", [False, True])
def test_compiled_stage_sets(wake, noise, lrw):
    counts = [700, 257, 5000]
    rng = np.random.default_rng(9)
    n = int(np.sum(counts))
    parts = configs.gaussian_bunch(n, 10)
    draws = rng.standard_normal((4, 5 * n))
    lost = (rng.random(n) < 0.02).astype(np.int32) * 2
    outs = []
    for n_rf, flush in ((1, True), (1, False), (2, True)):
        ring, secs, _ = configs.lattice()
        q, ne = configs.bunch_scalars(counts, ring)
        assert ring.n_rf == 1
        ring.n_rf = n_rf
        if n_rf == 2:
            ring.rf_vr[1] = ring.rf_vi[1] = 0.0
            ring.rf_harm[1] = ring.rf_harm[0]
        print(f"{n_rf} rf, wake {wake}, noise {noise}, long range {lrw}, flush {flush}", flush=True)
        tr = Tracker(ring, secs)
        tr.set_bunches(counts, q, ne, configs.train_gaps(3, 1, ring.harmonic))
        tr.upload(parts, lost)
        if wake is not None:
            tr.set_wake(50, wake, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
        if noise:
            tr.set_synrad(True, noise, 5)
        if lrw:
            tr.set_lrwake(2, [[0.01, 0.01, 100.0, 5.0, 5.0, 1, 3.5e7]])
        for t in range(4):
            if noise == 1:
                tr.push_noise(draws[t])
            tr.turn(t)
            if t == 1 and flush:
                tr.flush()
        outs.append((tr.download(), tr.wake_state()[0] if wake is not None else np.zeros(1)))
        tr.close()
    d0, h0 = outs[0]
    for k, (d1, h1) in enumerate(outs[1:]):
        assert np.array_equal(d0["lost"], d1["lost"]) and np.array_equal(h0, h1)
        for c in COORDS:
            if noise is None or k == 0:
                assert np.array_equal(d0[c], d1[c]), c
            else:
                same_but_for_fusing(d0[c], d1[c])


def same_but_for_fusing(a, b, turns=4):
    """Two sets that fuse roundings of the radiation stage differently: at most
    four a turn, each half an ulp of the scale and carried on in full by the
    maps (twice: through the other variable of its plane)."""
    assert np.max(np.abs(a - b)) <= turns * 4 * 2 * 2.0 ** -53 * np.max(np.abs(a))


@pytest.mark.parametrize("lrw", [False, True])
def test_compiled_beam_loading_set(lrw):
    """The set with a beam-loaded cavity against the general one, reached with
    an ideal cavity of voltage zero beside it."""
    counts = [700, 257, 5000]
    parts = configs.gaussian_bunch(int(np.sum(counts)), 11)
    lost = (np.random.default_rng(9).random(int(np.sum(counts))) < 0.02).astype(np.int32) * 2
    outs = []
    for n_rf in (0, 1):
        ring, secs, _ = configs.lattice()
        q, ne = configs.bunch_scalars(counts, ring)
        ring.n_rf = n_rf
        ring.rf_vr[0] = ring.rf_vi[0] = 0.0
        print(f"beam loading, {n_rf} rf, long range {lrw}", flush=True)
        tr = Tracker(ring, secs)
        tr.set_bunches(counts, q, ne, configs.train_gaps(3, 1, ring.harmonic))
        tr.upload(parts, lost)
        tr.set_wake(50, 1, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
        tr.set_synrad(True, 2, 5)
        if lrw:
            tr.set_lrwake(2, [[0.01, 0.01, 100.0, 5.0, 5.0, 1, 3.5e7]])
        tr.set_beam_loading(dict(nres=1, mode=[1], type=[1], harm=[1], cold=[0], rs=[5e6], q0=[2e4], coupling=[3.0],
                                 detune=[-2e4], vol=[configs.rf_voltage(configs.BASE)], phase=[0.0], nbins=60,
                                 nturns=4, excite=[0], dirfb=[0]))
        for t in range(4):
            tr.turn(t)
        outs.append((tr.download(), tr.wake_state()[0]))
        tr.close()
    (d0, h0), (d1, h1) = outs
    assert np.array_equal(d0["lost"], d1["lost"]) and np.array_equal(h0, h1)
    assert np.max(np.abs(d0["dp"] - parts["dp"])) > 1e-6
    for c in COORDS:
        same_but_for_fusing(d0[c], d1[c])
