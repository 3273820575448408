"""Read-out through the pinned slots (131072 spins each): what was put in comes back in every bit,
below one slot, at its edge, over more slots than worker threads, by replica and by slot, from
several contexts that hand the buffers on and from threads that read one context at a time."""
import threading

import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,R", [(2, 1), (16, 31), (16, 32), (16, 33), (21, 125)])
def test_spins_come_back(L, R):
    from espins_amd.engine import Engine
    print(L, R, flush=True)
    m = Lt.cubic_model("sc", L, J=(1.0,))
    x = Lt.random_spins(m.N, R, 3, m.mag)
    with Engine(0) as other:                       # keeps the buffers alive between the two contexts
        other.set_model(m)
        for k in range(2):
            with Engine(0) as eng:
                eng.set_model(m)
                eng.set_replicas(np.linspace(0.5, 2.0, R), x)
                assert np.array_equal(eng.spins(), x)
                eng.run(6, measure=True, exchange=True, seed=5 + k)
                y, slot_rep = eng.spins(), np.asarray(eng.pt_map()[0]) - 1
                if sorted(slot_rep) == list(range(R)):
                    assert np.array_equal(eng.spins(by_slot=True), y[slot_rep])
                e = eng.energy_get()
                got = [None] * 6

                def read(i):
                    got[i] = (eng.spins(), eng.energy_get(), eng.stats()["acc"])

                th = [threading.Thread(target=read, args=(i,)) for i in range(len(got))]
                [t.start() for t in th]
                [t.join() for t in th]
                for s, en, acc in got:
                    assert np.array_equal(s, y) and np.array_equal(en, e) and np.array_equal(acc, got[0][2])
