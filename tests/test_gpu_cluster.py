"""Replicas shared by clusters of blocks (the automatic path of middle-sized models) against the
launch-per-colour path on the same inputs: plain and tempering schedules, both proposals, bonds of
every kind, per-bond couplings, uneven parts, one replica and as many as two CUs each hold, the
trace, runs split over several launches, and changes between the two paths in one context.

Same counters, same order of updates: decisions differ only where dE's rounding (about z 1e-16)
straddles a uniform, so spins, counts and the replica map are equal and sums agree to rounding."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from espins_amd import setup_gen as Sg

pytestmark = pytest.mark.gpu


def run(m, tems, path, **kw):
    from espins_amd.engine import Engine
    with Engine(0) as eng:
        eng.set_path(path)
        eng.set_model(m)
        eng.set_replicas(tems, Lt.random_spins(m.N, len(tems), 7, m.mag))
        eng.set_trace(64)
        eng.run(kw.pop("rounds"), measure=True, seed=21, tilt=0.3, **kw)
        st = eng.stats()
        assert np.allclose(st["e_run"], eng.energy_get(), rtol=1e-11, atol=1e-9)
        return st, eng.spins(), eng.pt_map(), eng.trace()


def same(a, b):
    assert np.array_equal(a[0]["rejected"], b[0]["rejected"]) and a[0]["nmeas"] == b[0]["nmeas"]
    assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
    assert np.allclose(a[1], b[1], rtol=0, atol=1e-13)
    assert np.allclose(a[0]["acc"], b[0]["acc"], rtol=1e-11)
    assert np.allclose(a[3], b[3], rtol=1e-11)


CASES = [
    ("fcc", 8, dict(J=(-1.0, 0.2, 0.05), K=-0.1), 8), ("sc", 12, dict(J=(1.0,), B=0.1, D=0.3), 13),
    ("bcc", 9, dict(J=(1.0, -0.2), field=0.4), 64), ("fcc", 7, dict(J=(1.0,), B=0.05), 5),
    ("sc", 16, dict(J=(1.0, 0.3)), 1), ("sc", 14, dict(J=(1.0,)), 128),
]


@pytest.mark.parametrize("kind,L,kw,R", CASES)
@pytest.mark.parametrize("mode,exchange", [("random", True), ("const", False)])
def test_clusters_equal_phases(kind, L, kw, R, mode, exchange):
    print(kind, L, kw, R, mode, exchange, flush=True)
    m = Lt.cubic_model(kind, L, **kw)
    tems = np.linspace(0.4, 2.5, R)
    args = dict(rounds=5, steps_per_round=2, steps_measure=1 + (R % 2), mode=mode, exchange=exchange)
    same(run(m, tems, 0, **args), run(m, tems, 1, **args))


def test_clusters_with_per_bond_couplings():
    m = Lt.cubic_model("sc", 15, J=(1.0,))
    m.J = Sg.spin_glass(m.J, np.full((m.J.z, m.N), 0.8), 99)
    tems = np.linspace(0.3, 1.5, 11)
    args = dict(rounds=6, mode="random", exchange=True)
    same(run(m, tems, 0, **args), run(m, tems, 1, **args))


def test_change_of_path_and_sweeps_over_several_launches():
    from espins_amd.engine import Engine
    m = Lt.cubic_model("sc", 12, J=(1.0,))
    tems = np.linspace(0.5, 2.0, 4)
    out = []
    for paths in ((0, 1, 0), (1, 1, 1)):
        with Engine(0) as eng:
            eng.set_model(m)
            eng.set_replicas(tems, Lt.random_spins(m.N, 4, 5))
            sw = 0
            for p, n in zip(paths, (7, 3, 140000)):      # the last: more phases than one launch takes
                eng.set_path(p)
                eng.sweep(n, mode="random", seed=3, sweep0=sw)
                sw += n
            st = eng.stats()
            # the running energy adds 140010 sweeps of differences: 5e8 roundings of 1e-16 relative
            assert np.allclose(st["e_run"], eng.energy_get(), rtol=1e-9, atol=1e-7)
            out.append((st["rejected"], eng.spins()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.allclose(out[0][1], out[1][1], rtol=0, atol=1e-13)
