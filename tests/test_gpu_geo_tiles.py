"""Colour phases on tiles of one geometry group (bond lists sorted by shift, computed partners,
scalar coefficients) against the same sweeps through the explicit tables, and the per-wave sums
against direct sums, at the tile edges: groups of 8 sites (tables), 27, 64 (one full tile), 125
and 343 sites (uneven tiles and runs with spare waves), bonds of every kind, padded slots.

Both paths add a site's bonds in a different order, so dE differs by about z eps |J| ~ 1e-14;
a decision flips with probability ~1e-14 per update and the proposals do not depend on dE, so
spins agree to the rounding of the proposal itself (1e-15) and counts exactly."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu

CASES = [
    ("sc", 4, dict(J=(1.0,))), ("sc", 6, dict(J=(1.0, 0.3), field=0.4)), ("sc", 8, dict(J=(1.0,), B=0.1, D=0.3)),
    ("sc", 14, dict(J=(1.0,), D=0.2, K=0.1)), ("bcc", 9, dict(J=(1.0, -0.2))), ("bcc", 10, dict(J=(-1.0, 0.2), B=0.1)),
    ("fcc", 6, dict(J=(-1.0, 0.2, 0.05), K=-0.1)), ("fcc", 7, dict(J=(1.0,))), ("fcc", 15, dict(J=(1.0, -0.2), B=0.05)),
]


@pytest.mark.parametrize("mode", ["random", "const"])
@pytest.mark.parametrize("kind,L,kw", CASES)
def test_geometry_tiles_equal_tables(kind, L, kw, mode):
    from espins_amd.engine import Engine
    print(kind, L, kw, mode, flush=True)
    m = Lt.cubic_model(kind, L, **kw)
    tems = np.linspace(0.4, 2.0, 9)
    got = []
    for indexing in (0, 1):
        with Engine(0) as eng:
            eng.set_path(1)
            eng.set_model(m)
            eng.set_indexing(indexing)
            eng.set_replicas(tems, Lt.random_spins(m.N, 9, 3))
            eng.run(4, steps_per_round=2, measure=True, exchange=True, mode=mode, tilt=0.3, seed=9)
            st = eng.stats()
            s = eng.spins()
            assert np.allclose(st["e_run"], eng.energy_get(), rtol=1e-11, atol=1e-9)
            got.append((st, s, eng.pt_map()))
    (a, sa, ma), (b, sb, mb) = got
    assert np.array_equal(a["rejected"], b["rejected"])
    assert np.array_equal(ma[0], mb[0]) and np.array_equal(ma[1], mb[1])
    # 8 sweeps of cone proposals rotate a spin from its old direction: errors add up, ~8 x 1e-15
    assert np.allclose(sa, sb, rtol=0, atol=1e-13)
    assert np.allclose(a["acc"], b["acc"], rtol=1e-11)
    assert a["nmeas"] == 8
