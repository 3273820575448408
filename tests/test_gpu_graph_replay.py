"""A measurement after a replayed round sees the spins that the replay left: a captured round is
replayed after sweeps of another kind in the same context -- plain after learned, learned after
plain -- on the launch-per-colour path, whose phases leave spin sums, and on the LDS path, which
leaves none."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from espins_amd import learn as Ln

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [1, 2])
@pytest.mark.parametrize("captured,between", [("random", "learned"), ("learned", "random"), ("const", "random"),
                                              ("learned", "learned")])
@pytest.mark.parametrize("how", ["sweep", "run"])
def test_measure_after_replay(path, captured, between, how):
    from espins_amd.engine import Engine
    print(path, captured, between, how, flush=True)
    R = 5
    m = Lt.cubic_model("sc", 6, J=(1.0, 0.1), B=0.05, K=-0.1)
    with Engine() as eng:
        eng.set_path(path)
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.3, 2.0, R), Lt.random_spins(m.N, R, 9, m.mag))
        eng.learn_set_weights(Ln.init_weights(5, out_scale=0.3))
        args = dict(measure=True, exchange=False, mode=captured, seed=3, graph=True)
        eng.run(1, **args)                                       # captures the round
        if how == "sweep":
            eng.sweep(2, mode=between, seed=4, sweep0=50)
        else:
            eng.run(2, measure=False, exchange=False, mode=between, seed=4, sweep0=50, graph=False)
        eng.run(3, sweep0=100, **args)                           # the same key: replays it
        eng.reset_stats()
        eng.measure()
        acc = eng.stats()["acc"]
        mag = np.linalg.norm(eng.spins(by_slot=True).mean(1), axis=1)
        e = eng.energy_get()
    # sums of N terms of size 1 in another order: below N eps / N of a mean
    np.testing.assert_allclose(acc[:, 3], mag, rtol=0, atol=1e-13)
    np.testing.assert_allclose(acc[:, 4], mag**2, rtol=0, atol=1e-13)
    np.testing.assert_allclose(acc[:, 0], e, rtol=1e-11, atol=1e-9)
