"""Clusters of blocks after a change of the replica count in one context: a block's LDS grows with
the replicas, so tables of the same number of parts may serve one count and not the next."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from espins_amd.engine import plan_clusters

LDS = 160 * 1024


def test_plan_depends_on_the_replica_count():
    m = Lt.cubic_model_fast("sc", 22, J=(1.0,))
    few, many = plan_clusters(m, 90), plan_clusters(m, 128)
    assert few["parts"] == 2 and few["lds"] <= LDS < few["lds"] + 120 * (128 - 90)
    assert many["parts"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [(90, 128, 90), (128, 90, 5)])
def test_replica_counts_in_one_context(counts):
    from espins_amd.engine import Engine
    m = Lt.cubic_model_fast("sc", 22, J=(1.0,))
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            for R in counts:
                print(path, R, flush=True)
                eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 3))
                eng.run(4, measure=True, exchange=True, seed=8)
                parts = plan_clusters(m, R)["parts"] if path == 0 else 0
                assert eng.cluster_info()["sweeps"] == (4 if parts else 0)
                if path == 0:
                    assert eng.cluster_info()["parts"] == parts
                out.append((eng.stats(), eng.spins(), eng.pt_map()))
    for a, b in zip(out[:len(counts)], out[len(counts):]):
        assert np.array_equal(a[0]["rejected"], b[0]["rejected"])
        assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
        # same decisions; sums of N z terms of size 1 in another order
        np.testing.assert_allclose(a[1], b[1], rtol=0, atol=1e-13)
        np.testing.assert_allclose(a[0]["acc"], b[0]["acc"], rtol=1e-11)
