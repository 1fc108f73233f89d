"""The long-range sum at the edges of its split (16 waves over the turns, 64
lanes over the bunches): one bunch, a wave's bunches and one more, fewer and
more turns than waves, until the history has filled and come round.  Kicks
against the oracle within 1e-10 of the largest, as the other long-range tests
(of a single bunch's first turn there is no kick), the recorded means against
the moments exactly."""
import numpy as np
import pytest

import oracle as O
from test_gpu_lrwake import lrw_cfg
from test_gpu_train import setup_train

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nturns", [(1, 2), (3, 33), (64, 16), (65, 17), (130, 2)])
def test_split_of_the_long_range_sum(nb, nturns):
    counts = [40 + b % 3 for b in range(nb)]
    ring, secs, counts, gap, q, ne, cfg, tr, bunches, off = setup_train(counts, 17)
    c = lrw_cfg(secs, nturns)
    tr.set_lrwake(c["nturns"], c["sectors"], c["res"], c["beta_x"], c["beta_y"])
    tr.set_history(nturns + 2)
    ot = O.OracleTrain(ring, secs[0], counts, ne, gap, None, 1, lrw=c)
    print(f"long-range sum of {nb} bunches, {nturns} turns", flush=True)
    for t in range(nturns + 2):
        tr.turn(t)
        ot.turn(bunches, t)
        k, ok = tr.lrwake_kick(), ot.last_lrw_kick
        for pl in range(3):
            scale = np.max(np.abs(ok[:, pl]))
            assert scale > 0 or (t == 0 and nb == 1)
            np.testing.assert_allclose(k[:, pl], ok[:, pl], rtol=0, atol=1e-10 * scale)
    m, h = tr.moments(), tr.history(nturns + 1, 1)
    for b in range(nb):
        assert np.array_equal(h[b]["mean"][[1, 3]], m[b]["mean"][[1, 3]])
    tr.close()


@pytest.mark.parametrize("nb,nturns", [(150, 1), (150, 3), (90, 5), (70, 7), (64, 9)])
def test_several_waves_for_a_turn(nb, nturns):
    """Fewer turns than half the waves: the bunches of a turn over the lanes
    of several waves, with waves left over, in blocks of 4 to 16 waves."""
    test_split_of_the_long_range_sum(nb, nturns)
