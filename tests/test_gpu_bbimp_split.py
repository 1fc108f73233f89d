"""The broadband impedance at the edges of its split: bunches of one
macroparticle and around a binning block's share, ranges of bins with many
copies of the LDS window, one, or several windows, macroparticles lost in the
turn far outside the survivors' range, profiles over several smoothing tiles
and voltages over several tiles of sources, in both methods.  Profiles and
voltages against numpy on the same coordinates (a turn without radiation
leaves z, x and y as binned: counts exactly, sums of up to 1e4 terms within
1e-12 of the largest value), kicks against the difference to a twin without
the impedance, within the last digits of the momenta."""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.tracker import Tracker

import oracle as O

pytestmark = pytest.mark.gpu

BETA = (5.0, 3.0)


def smooth(p):
    """gsl_filter_gaussian (51 taps, alpha 10, end values padded), rescaled."""
    t = np.exp(-0.5 * 100.0 * (np.arange(-25, 26) / 25.0) ** 2)
    y = np.convolve(np.pad(p, 25, mode="edge"), t / t.sum(), mode="valid")
    return y * (p.sum() / y.sum())


def run(ring, secs, counts, parts, setup):
    q, ne = configs.bunch_scalars(counts, ring)
    tr = Tracker(ring, secs)
    nb = len(counts)
    tr.set_bunches(counts, q, ne, configs.train_gaps(nb, 1, ring.harmonic) if nb > 1 else None)
    tr.upload(parts)
    out = []
    if setup:
        setup(tr)
    tr.turn(0)
    if setup:
        out = tr.bbimp_wake()
    d = tr.download()
    tr.close()
    return d, out, q


@pytest.mark.parametrize("td", [True, False])
@pytest.mark.parametrize("step,stretch,counts", [
    (5.0e-4, 1.0, [1, 4095, 4097, 9000]), (1.5e-4, 4.0, [6000, 255]), (2.0e-5, 1.0, [5000]),
    (1.2e-5, 1.5, [40_001, 300])])
def test_split(td, step, stretch, counts):
    if not td:
        step = max(step, 6.0e-5)  # at most 16383 bins
    ring, secs, _ = configs.lattice()
    n = int(np.sum(counts))
    off = np.concatenate([[0], np.cumsum(counts)])
    parts = configs.gaussian_bunch(n, 21)
    rng = np.random.default_rng(22)
    for b in range(len(counts)):
        parts["z"][off[b]:off[b + 1]] *= stretch
        parts["x"][off[b]:off[b + 1]] += 4e-5 * (b + 1)
        parts["y"][off[b]:off[b + 1]] -= 2e-5 * (b + 1)
        if counts[b] > 100:  # lost at this turn's marking, but counted by the impedance
            k = off[b] + rng.choice(counts[b], 5, replace=False)
            parts["y"][k] = 0.05
            parts["py"][k] = 0.0
            parts["z"][k] = [-0.2, 0.2, 0.21, 0.19, 0.0]
    print(f"td {td}, step {step}, {counts}", flush=True)
    flags = (1, 1, 1, 1, 1)
    if td:
        pos = np.arange(301) * step
        wakes = [a * np.exp(-pos / (60 * step)) * np.cos(pos / (20 * step) + ph)
                 for a, ph in ((1e15, 0.0), (2e16, 0.5), (-3e16, 1.0), (1e16, 0.2), (4e16, 1.5))]
        d, (V, pr), q = run(ring, secs, counts, parts, lambda t: t.set_bbimp_td(pos, wakes, beta=BETA))
        length = ring.t0 / ring.harmonic * configs.C_LIGHT
        dz = pos[1] - pos[0]
        nbin, zmin, half = int(length / dz), -length / 2, 0.0
    else:
        fmax = configs.C_LIGHT / (2 * step)
        nimp = int(0.45 / step)
        f = np.arange(nimp) / (nimp - 1.0)
        z = 1e4 / (1 + 1j * (f - 0.3))
        zt = [(s * z).real.copy() for s in (1.0, 2e2, 3e2, 1e2, -2e2)], [(s * z).imag.copy()
                                                                        for s in (1.0, 2e2, 3e2, 1e2, -2e2)]
        pl = [(zt[0][k], zt[1][k]) for k in range(5)]
        d, (V, pr), q = run(ring, secs, counts, parts, lambda t: t.set_bbimp(
            pl[0][0], pl[0][1], fmax, flags=flags, zdx=pl[1], zdy=pl[2], zqx=pl[3], zqy=pl[4], beta=BETA))
        dz = configs.C_LIGHT * ring.rbeta / (2 * fmax)
        nbin, zmin, half = 2 * nimp - 1, -dz * (nimp - 1), dz / 2
        length = ring.t0 / ring.harmonic * configs.C_LIGHT
        i0 = int((-length / 2 - zmin + dz / 2) / dz)
        i1 = int((length / 2 - zmin + dz / 2) / dz)
    assert V.shape[2] == nbin
    twin, _, _ = run(ring, secs, counts, parts, None)
    assert (d["lost"] != 0).sum() == 5 * sum(c > 100 for c in counts)
    for c in ("x", "y", "z", "lost"):
        assert np.array_equal(d[c], twin[c]), c
    for b in range(len(counts)):
        s = slice(off[b], off[b + 1])
        pos_b = (d["z"][s] - zmin + half) / dz
        assert np.min(np.abs(pos_b - np.rint(pos_b))) > 1e-11
        k = np.trunc(pos_b).astype(int)
        cnt = np.bincount(k, minlength=nbin).astype(float)
        sx, sy = (np.bincount(k, weights=d[c][s], minlength=nbin) for c in ("x", "y"))
        charge = q[b] * configs.E_CHARGE
        if td:
            rho = smooth(cnt * charge)
            avg = [np.divide(v, cnt, out=np.zeros(nbin), where=cnt > 0) for v in (sx, sy)]
            prof = [rho] + avg
            src = [rho, rho * avg[0], rho * avg[1], rho, rho]
            want = [-np.convolve(src[p][::-1], wakes[p])[:nbin][::-1] for p in range(5)]
        else:
            prof = []
            for v in (cnt, sx, sy):
                v = v * (charge / dz * configs.C_LIGHT)
                v[i0:i1] = smooth(v[i0:i1])
                prof.append(v)
            src = [prof[0], prof[1], prof[2], prof[0], prof[0]]
            want = []
            for p in range(5):
                zz = pl[p][0] + 1j * pl[p][1]
                spec = np.fft.rfft(src[p]) * (zz if p == 0 else 1j * zz)
                spec[0] = spec[0].real
                want.append((-1 if p == 0 else 1) * np.fft.irfft(spec, nbin))
        for r in range(3):
            np.testing.assert_allclose(pr[r][b], prof[r], rtol=0, atol=1e-12 * np.max(np.abs(prof[r])))
        for p in range(5):
            np.testing.assert_allclose(V[p][b], want[p], rtol=0, atol=1e-11 * np.max(np.abs(want[p])))
        kk = V[:, b, :] / ring.energy / ring.rbeta ** 2
        x, y = d["x"][s], d["y"][s]
        exp = dict(dp=kk[0][k], px=(kk[1][k] + kk[3][k] * x) / BETA[0], py=(kk[2][k] + kk[4][k] * y) / BETA[1])
        for c, v in exp.items():
            assert np.max(np.abs(v)) > 1e-9 * np.max(np.abs(twin[c][s]))
            tol = 1e-12 * np.max(np.abs(v)) + 4e-16 * np.max(np.abs(twin[c][s]))
            assert np.max(np.abs(d[c][s] - twin[c][s] - v)) <= tol, c
