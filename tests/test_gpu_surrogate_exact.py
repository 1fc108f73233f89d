"""Electrons that the learned field leaves to the exact one, next to the centre
of the cloud, against the field's expansion there.  The field of a Gaussian
beam of sizes (sx, sy) per unit line charge is
F_x = -x int_0^inf exp(-x^2/(a + q) - y^2/(b + q)) (a + q)^-3/2 (b + q)^-1/2 dq,
a = 2 sx^2, b = 2 sy^2 (the round beam's (1 - exp(-r^2/a))/r^2 follows); two
terms of the exponential leave 1e-19 / max(sx, sy) for offsets up to 2e-4 sizes.
w(z) of order one cancels to a field of 1e-4 / max(sx, sy) there, so the error is
that of w(z): by the general w(z) 1.4e-16 / max(sx, sy) rms, by the plain kick's
rational approximation 1.0e-15 (both formulas compiled for the CPU, against 40
digits); the bound lies halfway between in the logarithm."""
import numpy as np
import pytest

from cetasim_amd import configs
from cetasim_amd.surrogate import Surrogate
from cetasim_amd.tracker import Tracker

pytestmark = pytest.mark.gpu

R_E = 2.81794092e-15  # classical electron radius as the reference has it


def test_kicks_next_to_the_centre():
    p = configs.BASE
    ring, secs, _ = configs.lattice(p)
    n, m = 4000, 600
    parts = configs.gaussian_bunch(n, 21, p)
    rng = np.random.default_rng(4)
    off = 10 ** rng.uniform(np.log10(2e-5), np.log10(2e-4), (2, m)) * rng.choice([-1.0, 1.0], (2, m))
    for c in ("x", "px", "y", "py"):
        parts[c][:m] = 0.0
    q, ne = configs.bunch_scalars(np.array([n]), ring, p)
    ions = dict(mass_number=[28.0], cross_section=[2.0e-22], pressure=[1.0e-5], temperature=300.0, n_new=500,
                max_ions=10_000, loss_boundary=10.0, seed=6)
    sur = Surrogate()
    sur.generate(1 << 12, 1 << 10, 4)
    sur.init_params(7)
    tr = Tracker(ring, secs)
    # the cloud's centre moves a little with the electrons put next to it
    for _ in range(10):
        tr.set_bunches([n], q, ne)
        tr.upload(parts)
        tr.set_ions(configs.ion_config(ring, ions, p))
        tr.set_field_model(sur, 2)
        print("kick next to the cloud's centre", flush=True)
        tr.ion_phase(0)
        _, mx, my, sx, sy, charge = tr.ion_passages()[0, 0]
        dx, dy = parts["x"][:m] - mx, parts["y"][:m] - my
        near = np.abs(dx) / sx + np.abs(dy) / sy
        if near.max() < 5e-4:
            break
        parts["x"][:m], parts["y"][:m] = mx + off[0] * sx, my + off[1] * sy
    assert 1e-5 < near.min() and near.max() < 5e-4
    got = tr.download()
    tr.close()
    sur.close()
    ld = np.longdouble
    s, t = (ld(2) ** 0.5 * ld(v) for v in (sx, sy))
    dx, dy = dx.astype(ld), dy.astype(ld)

    def field(x, y, s, t):
        return -x * (2 / (s * (s + t)) - x * x * (2 * (2 * s + t) / (3 * s ** 3 * (s + t) ** 2))
                     - y * y * (2 / (s * t * (s + t) ** 2)))

    scale = 2 * charge * R_E / ring.rgamma
    size = max(sx, sy)
    err = np.hypot(got["px"][:m] / scale - field(dx, dy, s, t), got["py"][:m] / scale - field(dy, dx, t, s)) * size
    rms = float(np.sqrt(np.mean(err ** 2)))
    print(f"error of the exact kicks times the larger size: rms {rms:.2e}, largest {float(err.max()):.2e}")
    assert rms <= 3.7e-16
