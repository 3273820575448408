"""The magnetisation that a step measures from its phases' per-wave sums equals the spins' own,
while plain and learned steps alternate in one context (each keeps sums of its own), for colours
that fill their last wave and colours that do not, and more replicas than a block has threads."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from espins_amd import learn as Ln

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,R", [("sc", 5, 3), ("fcc", 6, 65), ("sc", 16, 8), ("fcc", 14, 64), ("sc", 4, 300)])
@pytest.mark.parametrize("graph", [False, True])
def test_measured_magnetisation(kind, L, R, graph):
    from espins_amd.engine import Engine
    print(kind, L, R, graph, flush=True)
    m = Lt.cubic_model(kind, L, J=(1.0, 0.1), B=0.05, K=-0.1)
    with Engine() as eng:
        eng.set_path(1)
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.3, 2.0, R), Lt.random_spins(m.N, R, 9, m.mag))
        eng.set_trace(16)
        eng.run(1, measure=True, exchange=False, seed=3, graph=graph)      # before there are weights
        eng.learn_set_weights(Ln.init_weights(5, out_scale=0.3))
        mags = [np.linalg.norm(eng.spins(by_slot=True).mean(1), axis=1)]
        es = [eng.energy_get()]
        for k, mode in enumerate(["learned", "random", "learned", "const", "learned"]):
            eng.run(1, measure=True, exchange=False, mode=mode, seed=4 + k, graph=graph)
            mags.append(np.linalg.norm(eng.spins(by_slot=True).mean(1), axis=1))
            es.append(eng.energy_get())
        t = np.asarray(eng.trace())
    assert t.shape == (6, R, 2)
    # sums of N terms of size 1 in another order: below N eps / N of a mean
    np.testing.assert_allclose(t[:, :, 1], mags, rtol=0, atol=1e-13)
    np.testing.assert_allclose(t[:, :, 0], es, rtol=1e-11, atol=1e-9)
