"""A bunch of more segments than the closing kernels read themselves (2048):
their partial sums folded in groups of 256 first.  Bunches on both sides of the
bound and without a whole group, over the wakes, against a layout of few
segments: coordinates, loss codes, bins and z ranges equal on the fixed grid
(or without a wake); moments, and the reference's edges, within the rounding of
regrouped sums of n terms (1e-12 of the sizes they are made of)."""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.tracker import COORDS, Tracker

pytestmark = pytest.mark.gpu

BBR = configs.BASE["bbr"]
SZ = configs.BASE["sig"][2]


@pytest.mark.parametrize("wake", [None, 0, 1])
@pytest.mark.parametrize("counts", [[512 * 2048 + 1], [300, 512 * 2300 + 7, 512 * 256, 1]])
def test_many_segments(counts, wake):
    ring, secs, _ = configs.lattice()
    n, nb = int(np.sum(counts)), len(counts)
    q, ne = configs.bunch_scalars(counts, ring)
    parts = configs.gaussian_bunch(n, 31)
    outs = []
    for layout in ((5, 0), (2**31 - 1, 512)):
        tr = Tracker(ring, secs)
        tr.set_bunches(counts, q, ne, configs.train_gaps(nb, 1, ring.harmonic) if nb > 1 else None)
        tr.upload(parts)
        if wake is not None:
            tr.set_wake(64, wake, -5 * SZ, 5 * SZ, BBR["rs"], BBR["q"], BBR["fr"])
        tr.set_lrwake(2, [[0.01, 0.01, 100.0, 5.0, 5.0, 1, 3.5e7]])
        tr.set_layout(*layout)
        tr.set_history(4)
        print(f"{counts} macroparticles, layout {layout}, wake {wake}", flush=True)
        tr.turn(0)
        first = tr.wake_state() if wake is not None else None
        tr.run_turns(1, 3)
        tr.flush()
        outs.append((first, tr.history(0, 4), tr.moments(), tr.download()))
        tr.close()
    (w0, h0, m0, d0), (w1, h1, m1, d1) = outs
    if wake == 0:
        # edges from the z range and rms of sums in another order
        np.testing.assert_allclose(w0[1], w1[1], rtol=1e-12)
        assert np.array_equal(w0[0].sum(axis=1), w1[0].sum(axis=1))
    if wake == 1:
        assert np.array_equal(w0[0], w1[0]) and np.array_equal(w0[1], w1[1])
    # with the long-range wake the kicks follow the centroids: equal to 1e-12
    # of the coordinates' scale after four turns
    for c in COORDS:
        assert np.max(np.abs(d0[c] - d1[c])) <= 1e-12 * np.max(np.abs(d0[c])), c
    assert np.array_equal(d0["lost"], d1["lost"])
    for a, b in zip(list(h0) + list(m0), list(h1) + list(m1)):
        assert a["n_alive"] == b["n_alive"] and a["loss_count"] == b["loss_count"]
        if a["n_alive"] < 2:
            continue
        sizes = np.sqrt(np.maximum(np.array([a["c2"][i] for i in (0, 2, 3, 5, 6, 8)]), 0.0))
        for i in range(6):
            assert abs(a["mean"][i] - b["mean"][i]) <= 1e-12 * sizes[i], i
        for k, (i, j) in enumerate(((0, 0), (0, 1), (1, 1), (2, 2), (2, 3), (3, 3), (4, 4), (4, 5), (5, 5))):
            assert abs(a["c2"][k] - b["c2"][k]) <= 1e-12 * sizes[i] * sizes[j], k
