"""Calls are synchronous at return: the statistics are cleared, not only queued to be, when
reset_stats comes back (the stream has nothing left to do)."""
import numpy as np
import pytest
import torch

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


def test_reset_stats_waits():
    from espins_amd.engine import Engine
    m = Lt.cubic_model("sc", 8, J=(1.0,))
    idle = []
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.5, 2.0, 64), Lt.random_spins(m.N, 64, 5))
        stream = torch.cuda.ExternalStream(eng.stream())
        for k in range(50):
            eng.run(1, seed=2, sweep0=k)
            eng.reset_stats()
            idle.append(stream.query())
        assert eng.stats()["nmeas"] == 0
    assert all(idle)
