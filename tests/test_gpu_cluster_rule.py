"""Which kernel serves replicas that one block holds: clusters of blocks where they are the faster one
(exchanges at every step or second step, many passes of a block over a colour, unmeasured sweeps), one
block per replica elsewhere (two colours with an exchange every third step; parts of more sites a colour
than a block has threads)."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,R,J,every,served", [
    ("sc", 12, 85, (1.0,), 1, True), ("sc", 12, 85, (1.0,), 2, True), ("sc", 12, 85, (1.0,), 3, False), ("bcc", 10, 128, (1.0,), 3, False),
    ("sc", 14, 48, (1.0,), 3, True), ("sc", 14, 48, (1.0, 0.3), 3, True), ("sc", 16, 48, (1.0,), 0, True), ("sc", 16, 85, (1.0,), 0, False),
    ("bcc", 12, 85, (1.0,), 5, False), ("bcc", 12, 100, (1.0,), 0, False), ("sc", 16, 85, (1.0, 0.3), 0, True), ("fcc", 10, 85, (1.0,), 5, True)])
def test_runs(kind, L, R, J, every, served):
    from espins_amd.engine import Engine
    print(kind, L, R, J, every, flush=True)
    m = Lt.cubic_model_fast(kind, L, J=J)
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.4, 2.0, R), Lt.random_spins(m.N, R, 3))
        assert eng.model_info()["lds"]
        n = 30
        if every:
            eng.run(n // every, steps_per_round=every, measure=True, exchange=True, seed=4)
        else:
            eng.run(1, steps_per_round=n, measure=True, exchange=False, seed=4, graph=False)
        assert eng.cluster_info()["sweeps"] == (n if served else 0)
        st = eng.stats()
        assert st["nmeas"] == n
        np.testing.assert_allclose(st["e_run"], eng.energy_get(), rtol=1e-11, atol=1e-9)
        if not every:
            eng.sweep(n, seed=4, sweep0=n)         # nothing measured: clusters
            assert eng.cluster_info()["sweeps"] == n
