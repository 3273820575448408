"""Clusters of few replicas in many parts (up to one per CU): block 0 adds the parts' sums with several
threads to a sum, where there are more than 16 -- odd numbers of parts, one replica and several."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,R", [("sc", 32, 1), ("sc", 24, 1), ("sc", 20, 3), ("sc", 25, 7), ("fcc", 12, 2), ("sc", 22, 15)])
def test_many_parts(kind, L, R):
    from espins_amd.engine import Engine
    print(kind, L, R, flush=True)
    m = Lt.cubic_model_fast(kind, L, J=(1.0,))
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 5))
            eng.set_trace(16)
            eng.run(6, steps_per_round=2, measure=True, exchange=R > 1, seed=12)
            if path == 0:
                info = eng.cluster_info()
                assert info["parts"] >= 16 and info["sweeps"] == 12
            out.append((eng.stats(), eng.pt_map(), eng.spins(), eng.trace(), eng.energy_get()))
    (a, ma, sa, ta, ea), (b, mb, sb, tb, _) = out
    assert np.array_equal(a["rejected"], b["rejected"]) and a["nmeas"] == b["nmeas"] == 12
    assert np.array_equal(ma[0], mb[0]) and np.array_equal(ma[1], mb[1])
    # same decisions; sums of N z terms of size 1 in another order
    np.testing.assert_allclose(sa, sb, rtol=0, atol=1e-13)
    np.testing.assert_allclose(a["acc"], b["acc"], rtol=1e-11)
    np.testing.assert_allclose(ta, tb, rtol=1e-11)
    np.testing.assert_allclose(a["e_run"], ea, rtol=1e-11, atol=1e-9)
