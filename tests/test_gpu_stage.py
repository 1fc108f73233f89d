"""The particle state's way to the host at the edges of its stretches (65 536
macroparticles, a ring of two, a block of 256): every coordinate and loss code
as uploaded, bit for bit, also into some of the arrays alone, again, and after
the handle's bunches grew or shrank."""
import numpy as np
import pytest

from cetasim_amd import capi, configs
from cetasim_amd.tracker import COORDS, Tracker

pytestmark = pytest.mark.gpu


def test_download_at_the_edges_of_a_stretch():
    ring, secs, _ = configs.lattice()
    tr = Tracker(ring, secs)
    rng = np.random.default_rng(5)
    for counts in ([1], [257, 255], [65_535], [65_537], [131_072], [70_000, 61_073], [300], [700_001]):
        n = int(np.sum(counts))
        print(f"download of {counts}", flush=True)
        q, ne = configs.bunch_scalars(counts, ring)
        tr.set_bunches(counts, q, ne, configs.train_gaps(len(counts), 1, ring.harmonic) if len(counts) > 1 else None)
        parts = {c: rng.standard_normal(n) for c in COORDS}
        lost = rng.integers(0, 3, n).astype(np.int32)
        tr.upload(parts, lost)
        for _ in range(2):
            d = tr.download()
            assert all(np.array_equal(d[c], parts[c]) for c in COORDS) and np.array_equal(d["lost"], lost)
        some = {c: np.full(n, -7.0) for c in ("py", "z")}
        args = [capi.dptr(some[c]) if c in some else None for c in COORDS]
        capi.check(tr.lib.cts_download(tr.h, *args, None))
        assert all(np.array_equal(some[c], parts[c]) for c in some)
        only = np.full(n, -7, np.int32)
        capi.check(tr.lib.cts_download(tr.h, *[None] * 6, capi.i32ptr(only)))
        assert np.array_equal(only, lost)
        capi.check(tr.lib.cts_download(tr.h, *[None] * 7))
    tr.close()


def test_download_of_few_arrays():
    """One and two arrays on both sides of the sizes from which they are copied
    directly (131 072 and 262 144 macroparticles), with and without loss codes."""
    ring, secs, _ = configs.lattice()
    tr = Tracker(ring, secs)
    rng = np.random.default_rng(6)
    for n in (131_072, 131_073, 262_144, 262_145):
        print(f"few arrays of {n}", flush=True)
        q, ne = configs.bunch_scalars([n], ring)
        tr.set_bunches([n], q, ne)
        parts = {c: rng.standard_normal(n) for c in COORDS}
        lost = rng.integers(0, 3, n).astype(np.int32)
        tr.upload(parts, lost)
        for names in (("z",), ("x", "dp"), ("px", "lost"), ("y", "py", "lost")):
            out = {c: np.full(n, -7, np.int32 if c == "lost" else np.float64) for c in names}
            args = [capi.dptr(out[c]) if c in out else None for c in COORDS]
            capi.check(tr.lib.cts_download(tr.h, *args, capi.i32ptr(out["lost"]) if "lost" in out else None))
            for c in names:
                assert np.array_equal(out[c], lost if c == "lost" else parts[c]), c
    tr.close()
