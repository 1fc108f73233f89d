"""The default layouts of the streaming pass against an explicit one on the
same particles, at the edges of the rule that picks them (one bunch of less
or more than a block, few and many bunches, tiles for many particles):
coordinates, loss codes and bin counts bit-identical on the fixed grid,
means and second
moments to 1e-12 of the bunch's sizes (partial sums regrouped).  And the electron-side ion kick,
an item of up to 256 macroparticles per block, at the edges of its items."""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.tracker import COORDS, Tracker

import oracle as O
from test_gpu_train import BBR, ION_TEST, compare_coords, setup_train

pytestmark = pytest.mark.gpu

SZ = configs.BASE["sig"][2]


@pytest.mark.parametrize("counts", [[1], [255], [257], [200_001], [1, 300, 256], [3000] * 8, [9_001] * 90,
                                    [700, 3] * 60, [4_800_000, 5, 70_000]])
def test_default_layouts_agree(counts):
    ring, secs, _ = configs.lattice()
    counts = np.array(counts, np.int64)
    q, ne = configs.bunch_scalars(counts, ring)
    rng = np.random.default_rng(8)
    n = int(counts.sum())
    sx, sy, sz, sd = configs.BASE["sig"]
    scale = dict(x=sx, px=sx / 10, y=sy, py=sy / 10, z=sz, dp=sd)
    parts = {c: rng.standard_normal(n) * scale[c] for c in COORDS}
    lost = (rng.random(n) < 0.02).astype(np.int32) * 2
    lost[np.cumsum(counts) - counts] = 0  # every bunch keeps a particle
    print(f"default layout of {len(counts)} bunches, {n} macroparticles", flush=True)
    outs = []
    for lay in (None, (7, 0)):
        tr = Tracker(ring, secs)
        tr.set_bunches(counts, q, ne, configs.train_gaps(len(counts), 2, ring.harmonic))
        tr.upload(parts, lost)
        tr.set_wake(64, 1, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
        tr.set_synrad(True, 2, 3)
        if lay:
            tr.set_layout(*lay)
        for t in range(2):
            tr.turn(t)
        outs.append((tr.wake_state()[0], tr.moments(), tr.download()))
        tr.close()
    (h0, m0, d0), (h1, m1, d1) = outs
    assert np.array_equal(h0, h1) and h0.sum() > 0
    for c in COORDS + ("lost",):
        assert np.array_equal(d0[c], d1[c]), c
    for a, b in zip(m0, m1):
        assert a["n_alive"] == b["n_alive"] and a["zmin"] == b["zmin"] and a["zmax"] == b["zmax"]
        if a["n_alive"] > 1:
            sizes = np.sqrt(np.maximum([b["c2"][i] for i in (0, 2, 3, 5, 6, 8)], 0.0))
            assert np.all(np.abs(a["mean"] - b["mean"]) <= 1e-12 * sizes)
            pairs = ((0, 0), (0, 1), (1, 1), (2, 2), (2, 3), (3, 3), (4, 4), (4, 5), (5, 5))
            bound = np.array([1e-12 * sizes[i] * sizes[j] for i, j in pairs])
            assert np.all(np.abs(a["c2"] - b["c2"]) <= bound)


@pytest.mark.parametrize("nspec", [1, 2])
def test_ion_kick_items(nspec):
    counts = [255, 256, 257, 512, 700]
    ions = dict(ION_TEST, mass_number=[28.0, 18.0][:nspec], cross_section=[2.0e-22, 1.6e-22][:nspec],
                pressure=[1.0e-5, 0.4e-5][:nspec])
    ring, secs, counts, gap, q, ne, cfg, tr, bunches, off = setup_train(counts, 6, ions=ions, ne_scale=0.1)
    ot = O.OracleTrain(ring, secs[0], counts, ne, gap, cfg, ions["seed"])
    before = np.concatenate([b["px"] for b in bunches])
    print(f"ion kick items, {nspec} species", flush=True)
    tr.ion_phase(0)
    ot.ion_phase(bunches, 0)
    got = tr.download()
    compare_coords(got, bunches, off, 1e-12)
    assert np.max(np.abs(got["px"] - before)) > 1e-8 * np.max(np.abs(before))
    tr.close()


@pytest.mark.parametrize("nspec,n_new,nb", [(2, 3000, 40), (1, 17_000, 3)])
def test_cloud_of_many_waves(nspec, n_new, nb):
    """Clouds over several coarse survivor counts (256 waves each) and, with
    40 bunches, a compaction between two segments: the cloud in slot order."""
    ions = dict(ION_TEST, mass_number=[28.0, 18.0][:nspec], cross_section=[2.0e-22, 1.6e-22][:nspec],
                pressure=[1.0e-5, 0.4e-5][:nspec], n_new=n_new, max_ions=400_000)
    counts = [400 + 3 * (b % 5) for b in range(nb)]
    ring, secs, counts, gap, q, ne, cfg, tr, bunches, off = setup_train(counts, 14, ions=ions, ne_scale=0.1,
                                                                       gap=[2] * nb)
    ot = O.OracleTrain(ring, secs[0], counts, ne, gap, cfg, ions["seed"])
    print(f"cloud of {nspec} x {n_new * nb} ions", flush=True)
    tr.ion_phase(0)
    exp = ot.ion_phase(bunches, 0)
    got = tr.ion_passages()
    np.testing.assert_allclose(got[:, :nspec, 5], exp[:, :nspec, 0], rtol=1e-12)
    np.testing.assert_allclose(got[:, :nspec, 1:5], exp[:, :nspec, 1:5], rtol=1e-9, atol=1e-18)
    for sp in range(nspec):
        cloud, ec = tr.ion_cloud(sp), ot.cloud.species(sp)
        assert len(cloud["x"]) == len(ec["x"]) > 30_000
        for c in ("x", "y", "vx", "vy"):
            np.testing.assert_allclose(cloud[c], ec[c], rtol=1e-9, atol=1e-9 * np.max(np.abs(ec[c])))
    tr.close()


def test_default_layout_comes_back():
    """What the default layout reports restores it, for later bunches too."""
    ring, secs, _ = configs.lattice()
    tr = Tracker(ring, secs)

    def bunches(counts):
        q, ne = configs.bunch_scalars(counts, ring)
        tr.set_bunches(counts, q, ne, configs.train_gaps(len(counts), 2, ring.harmonic))
        return tr.layout()

    small, large = [3000] * 8, [300_000] * 20
    first, other = bunches(small), bunches(large)
    assert first != other
    bunches(small)
    tr.set_layout(7, 512)
    assert tr.layout() == (7, 512)
    tr.set_layout(*first)
    assert tr.layout() == first and bunches(large) == other
    tr.close()
