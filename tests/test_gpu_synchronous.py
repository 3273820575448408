"""Calls are synchronous at return: the statistics are cleared, not only queued to be, when
reset_stats comes back (the stream has nothing left to do)."""
import ctypes as C

import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


def test_reset_stats_waits():
    from espins_amd.engine import Engine
    hip = C.CDLL("libamdhip64.so.7")             # the runtime the library is linked against
    hip.hipStreamQuery.argtypes = [C.c_void_p]
    m = Lt.cubic_model("sc", 8, J=(1.0,))
    idle = []
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.5, 2.0, 64), Lt.random_spins(m.N, 64, 5))
        for k in range(50):
            eng.run(1, seed=2, sweep0=k)
            eng.reset_stats()
            idle.append(hip.hipStreamQuery(eng.stream()) == 0)
        assert eng.stats()["nmeas"] == 0
    assert all(idle)
