"""Rounds of more launches than a graph may hold are accepted with graph=True and give the results of
the same schedule launched directly."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


def test_long_round_of_a_context():
    from espins_amd.engine import Engine
    m = Lt.cubic_model("sc", 6, J=(1.0,))
    out = []
    for graph in (True, False):
        with Engine(0) as eng:
            eng.set_path(1)
            eng.set_model(m)
            eng.set_replicas([0.7, 1.5], Lt.random_spins(m.N, 2, 5))
            # 560000 launches: capturing so long a chain ended the process
            eng.run(1, steps_per_round=2, steps_measure=140000, measure=True, exchange=True, seed=4, graph=graph)
            out.append((eng.spins(), eng.stats()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1]["acc"], out[1][1]["acc"]) and out[0][1]["nmeas"] == 2


@pytest.mark.parametrize("steps,M", [(1, 2000), (1100, 2)])
def test_long_round_of_a_batch(steps, M):
    from espins_amd.engine import Batch
    out = []
    for graph in (True, False):
        with Batch(0) as b:
            for k, L in enumerate((4, 6)):
                m = Lt.cubic_model("sc", L, J=(1.0, 0.2))
                b.add_chain(m, [0.7, 1.5], Lt.random_spins(m.N, 2, 5 + k))
                b.set_chain_config(k, path=1, tps=1)
            b.commit()
            b.run(2, steps_per_round=steps, steps_measure=M, measure=True, exchange=True, seed=4, graph=graph)
            out.append([(b.spins(k), b.stats(k)["acc"]) for k in range(2)])
    for x, y in zip(*out):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])
