"""The two variants of the ion segment with the field surrogate, for clouds of
few and of many waves: the host's bound of the waves picks one, in a graph the
capacity, so the same turns with plain launches (few) and replayed with a
capacity of 800 000 ions (many) give the same cloud and momenta bit for bit."""
import numpy as np
import pytest

from cetasim_amd.surrogate import Surrogate

from test_gpu_train import ION_TEST, setup_train

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sur():
    s = Surrogate()
    s.generate(1 << 14, 1 << 10, 4)
    s.init_params(7)
    yield s
    s.close()


@pytest.mark.parametrize("nspec", [1, 2])
def test_few_and_many_waves(sur, nspec):
    ions = dict(ION_TEST, mass_number=[28.0, 18.0][:nspec], cross_section=[2.0e-22, 1.6e-22][:nspec],
                pressure=[1.0e-5, 0.4e-5][:nspec], n_new=500, max_ions=800_000)
    outs = []
    for graph in (False, True):
        _, _, _, _, _, _, _, tr, _, _ = setup_train([700, 257, 3000, 900], 6, ions=ions, ne_scale=0.1)
        tr.set_field_model(sur, 3)
        print(f"surrogate cloud, {nspec} species, graph {graph}", flush=True)
        tr.run_turns(0, 4, graph=graph)
        outs.append((tr.download(), [tr.ion_cloud(p) for p in range(nspec)]))
        tr.close()
    (d0, c0), (d1, c1) = outs
    assert all(np.array_equal(d0[c], d1[c]) for c in d0)
    for a, b in zip(c0, c1):
        assert len(a["x"]) > 0 and all(np.array_equal(a[c], b[c]) for c in ("x", "y", "vx", "vy"))
