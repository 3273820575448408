"""The LDS-resident sweep, whose halves of a block take turns where a colour fits in half a block,
against the launch-per-colour path: colours of exactly half a block and one site row more, odd
numbers of colours, several lanes per site, one colour, runs in several calls; and the automatic
path, which takes clusters for frequent exchanges of small replicas in long runs only.

Same counters and order of updates: spins, counts and the map are equal, sums agree to rounding."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


def run(m, R, path, calls, rounds, tps=0, **kw):
    from espins_amd.engine import Engine
    with Engine(0) as eng:
        eng.set_path(path)
        if tps:
            eng.set_tps(tps)
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.4, 2.5, R), Lt.random_spins(m.N, R, 7, m.mag))
        for k in range(calls):
            eng.run(rounds, measure=True, seed=21 + k, tilt=0.3, **kw)
        st = eng.stats()
        assert np.allclose(st["e_run"], eng.energy_get(), rtol=1e-11, atol=1e-9)
        return st, eng.spins(), eng.pt_map()


def same(a, b):
    assert np.array_equal(a[0]["rejected"], b[0]["rejected"]) and a[0]["nmeas"] == b[0]["nmeas"]
    assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
    assert np.allclose(a[1], b[1], rtol=0, atol=1e-13)
    assert np.allclose(a[0]["acc"], b[0]["acc"], rtol=1e-11)


CASES = [
    ("sc", 8, dict(J=(1.0,)), 5, 0), ("sc", 9, dict(J=(1.0, 0.2)), 3, 0), ("sc", 10, dict(J=(1.0,), D=0.2), 3, 0),
    ("bcc", 5, dict(J=(1.0, 0.1), B=0.1), 4, 2), ("fcc", 4, dict(J=(1.0,), K=-0.2), 4, 8), ("sc", 2, dict(J=(1.0,)), 9, 0),
    ("fcc", 6, dict(J=(1.0, 0.2)), 2, 1), ("bcc", 6, dict(J=(1.0,), field=0.3), 300, 4),
]


@pytest.mark.parametrize("kind,L,kw,R,tps", CASES)
@pytest.mark.parametrize("mode,exchange", [("random", True), ("const", False)])
def test_lds_equals_phases(kind, L, kw, R, tps, mode, exchange):
    print(kind, L, kw, R, tps, mode, exchange, flush=True)
    m = Lt.cubic_model(kind, L, **kw)
    args = dict(rounds=3, steps_per_round=2, steps_measure=1 + (R % 2), mode=mode, exchange=exchange, calls=2)
    same(run(m, R, 2, tps=tps, **args), run(m, R, 1, **args))


@pytest.mark.parametrize("L,rounds,steps", [(8, 128, 2), (8, 127, 2), (8, 8, 40), (6, 300, 1)])
def test_automatic_path_equals_lds(L, rounds, steps):
    print(L, rounds, steps, flush=True)
    m = Lt.cubic_model("sc", L, J=(1.0, 0.1))
    args = dict(rounds=rounds, steps_per_round=steps, mode="random", exchange=True, calls=2)
    same(run(m, 12, 0, **args), run(m, 12, 2, **args))
