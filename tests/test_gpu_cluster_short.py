"""Short calls -- a sweep or two, one step -- on a context that clusters of blocks serve: they take the
other paths (a cluster call costs more than the launches it replaces), longer ones the clusters, and a
mixture of both gives the results of the launch-per-colour path."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,R,J,colours", [("sc", 18, 5, (1.0,), 2), ("sc", 20, 9, (1.0, 0.3), 4), ("fcc", 12, 3, (1.0,), 4),
                                                ("sc", 14, 6, (1.0, 0.3), 4)])
def test_short_calls_take_the_other_paths(kind, L, R, J, colours):
    from espins_amd.engine import Engine
    print(kind, L, R, J, flush=True)
    m = Lt.cubic_model(kind, L, J=J)
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 5))
            assert eng.coloring()[0] == colours
            at = 0
            for n in (1, 4, 1, 1, 4):
                eng.sweep(n, seed=3, sweep0=at)
                at += n
                if path == 0 and (n == 1 or kind != "sc" or L > 14):     # (sc 14^3 fits one block)
                    assert eng.cluster_info()["sweeps"] == (0 if n == 1 else n)
            for k, n in enumerate((1, 4, 1)):
                eng.run(n, measure=True, exchange=True, seed=3, sweep0=at, step0=k, start_parity=1 + k % 2)
                at += n
                if path == 0:
                    assert eng.cluster_info()["sweeps"] == (0 if n == 1 else n)
            out.append((eng.stats(), eng.pt_map(), eng.spins(), eng.energy_get()))
    (a, ma, sa, ea), (b, mb, sb, _) = out
    assert np.array_equal(a["rejected"], b["rejected"]) and a["nmeas"] == b["nmeas"] == 6
    assert np.array_equal(ma[0], mb[0]) and np.array_equal(ma[1], mb[1])
    # same decisions; sums of N z terms of size 1 in another order
    np.testing.assert_allclose(sa, sb, rtol=0, atol=1e-13)
    np.testing.assert_allclose(a["acc"], b["acc"], rtol=1e-11)
    np.testing.assert_allclose(a["e_run"], ea, rtol=1e-11, atol=1e-9)
