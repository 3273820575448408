"""A batch of more state than one replica group holds: the groups' borders cut chains, and every
chain still reproduces a single context with its stream base (same kernel, same order: in every
bit up to the sums over waves)."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Rsc,Rfcc", [(116, 96), (150, 70), (3, 250)])   # 12.7, 13.5 and 14.0 million spins
def test_groups_cut_chains(Rsc, Rfcc):
    from espins_amd.engine import Batch, Engine, set_stream_base
    print(Rsc, Rfcc, flush=True)
    cs = [(Lt.cubic_model_fast("sc", 40, J=(1.0, -0.1)), Lt.ladder("log", 0.5, 2.5, Rsc)),
          (Lt.cubic_model_fast("fcc", 24, J=(1.0,)), Lt.ladder("log", 0.6, 2.0, Rfcc)),
          (Lt.cubic_model_fast("sc", 6, J=(1.0,)), Lt.ladder("log", 0.6, 2.0, 3))]
    init = [Lt.random_spins(m.N, len(t), 10 + k, m.mag) for k, (m, t) in enumerate(cs)]
    assert sum(x.size for x in init) * 8 > 288 << 20
    sched = dict(steps_per_round=2, steps_measure=1, measure=True, exchange=True, seed=77)
    with Batch() as b:
        for k, ((m, t), s) in enumerate(zip(cs, init)):
            b.add_chain(m, t, s)
            b.set_chain_config(k, 1, 1)
        b.commit()
        b.run(2, **sched)
        res = [(b.spins(k), b.stats(k), b.pt_map(k)) for k in range(len(cs))]
    for k, ((m, t), s) in enumerate(zip(cs, init)):
        with Engine() as eng:
            eng.set_path(1)
            eng.set_model(m)
            set_stream_base(eng, k << 16)
            eng.set_replicas(t, s)
            eng.run(2, **sched)
            assert np.array_equal(eng.spins(), res[k][0])
            assert np.array_equal(eng.stats()["rejected"], res[k][1]["rejected"])
            assert np.allclose(eng.stats()["acc"], res[k][1]["acc"], rtol=1e-12)
            assert np.array_equal(eng.pt_map()[1], res[k][2][1])
