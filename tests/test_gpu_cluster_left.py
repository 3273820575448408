"""Cluster launches that find their CUs taken: the run goes on from the sweep they reached on the other
paths -- before the first launch, between the steps of a round, within a step -- with the results of
the launch-per-colour path; the context then goes without clusters for 1, 2, 4, ... runs.  The limit
makes the launches leave as if other work held the CUs; every block exits normally."""
import threading

import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu
PHASES = 1 << 18


def same(a, b, tol):
    assert np.array_equal(a[0]["rejected"], b[0]["rejected"]) and a[0]["nmeas"] == b[0]["nmeas"]
    assert np.array_equal(a[1][0], b[1][0]) and np.array_equal(a[1][1], b[1][1])
    np.testing.assert_allclose(a[2], b[2], rtol=0, atol=1e-13)
    # running energies add up the differences of every accepted update, each rounded to 1e-16 of its size
    np.testing.assert_allclose(a[0]["acc"], b[0]["acc"], rtol=tol)
    np.testing.assert_allclose(a[0]["e_run"], a[3], rtol=tol, atol=1e-7)


def result(eng):
    return eng.stats(), eng.pt_map(), eng.spins(), eng.energy_get()


@pytest.mark.parametrize("rounds,steps,M,exchange,limit", [
    (4, 2, 1, True, 0), (3, 2, 12000, True, 1), (2, 1, 33000, True, 1), (1, 3, 33000, False, 3), (2, 2, 33000, True, 6),
    (1, 2, 66000, True, 1)])
@pytest.mark.parametrize("trace", [False, True])      # with a trace the phases take over, else the LDS path
def test_run_goes_on_from_where_clusters_left(rounds, steps, M, exchange, limit, trace):
    from espins_amd.engine import Engine
    print(rounds, steps, M, exchange, limit, trace, flush=True)
    m, R = Lt.cubic_model("fcc", 6, J=(1.0, 0.2)), 4
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas(np.linspace(0.6, 2.0, R), Lt.random_spins(m.N, R, 5))
            if trace or path == 1:
                eng.set_trace(8)
            if path == 0:
                # replicas of this size get their tables in a run that is long enough
                eng.run(256, measure=False, exchange=True, seed=9)
                assert eng.cluster_info()["sweeps"] == 256
                eng.set_cluster_limit(limit)
            else:
                eng.run(256, measure=False, exchange=True, seed=9)
            eng.run(rounds, steps_per_round=steps, steps_measure=M, measure=True, exchange=exchange, seed=12,
                    sweep0=1000, step0=256)
            if path == 0:
                info = eng.cluster_info()
                most, n = PHASES // eng.coloring()[0], rounds * steps
                need = n * -(-M // most) if M > most else -(-n // (most // M))
                if exchange or trace:        # (without exchanges the LDS path serves this size)
                    assert info["launches"] == min(limit, need) and info["skip"] == (limit < need)
                    assert (info["sweeps"] > 0) == (limit > 0) and (info["sweeps"] < n * M) == (limit < need)
            out.append(result(eng))
    same(*out, tol=1e-11 if M == 1 else 1e-9)


def test_sweeps_go_on_from_where_clusters_left():
    from espins_amd.engine import Engine
    m, R, n = Lt.cubic_model("sc", 15, J=(1.0,)), 3, 140000
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas([0.6, 1.0, 2.0], Lt.random_spins(m.N, R, 5))
            eng.set_trace(1)
            eng.set_cluster_limit(1)
            eng.sweep(n, seed=12)
            if path == 0:
                assert eng.cluster_info()["sweeps"] == PHASES // eng.coloring()[0]
            out.append(result(eng))
    same(*out, tol=1e-9)


def test_runs_without_clusters_after_one_that_they_left():
    from espins_amd.engine import Engine
    m, R = Lt.cubic_model("sc", 15, J=(1.0,)), 3
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas([0.6, 1.0, 2.0], Lt.random_spins(m.N, R, 5))
        eng.set_trace(1)
        served, skip = [], []
        for k in range(12):
            eng.set_cluster_limit(0 if k in (0, 2, 5) else -1)
            eng.run(2, measure=False, seed=3, sweep0=2 * k)
            served.append(eng.cluster_info()["sweeps"])
            skip.append(eng.cluster_info()["skip"])
        assert np.allclose(eng.stats()["e_run"], eng.energy_get(), rtol=1e-11, atol=1e-9)
    # left in runs 0, 2 and 5, each time for twice as many runs
    assert skip == [1, 0, 2, 1, 0, 4, 3, 2, 1, 0, 0, 0]
    assert served == [0] * 10 + [2, 2]


def test_contexts_of_two_threads():
    from espins_amd.engine import Engine
    m, R = Lt.cubic_model("fcc", 12, J=(1.0, 0.1)), 32
    got = {}

    def job(k, path=0):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas(np.linspace(0.6, 2.0, R), Lt.random_spins(m.N, R, 5))
            for i in range(20):
                eng.run(5, measure=True, exchange=True, seed=12, sweep0=5 * i, step0=5 * i, start_parity=1 + i % 2)
            got[k] = result(eng)

    threads = [threading.Thread(target=job, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    job("phases", 1)
    for k in range(3):
        same(got[k], got["phases"], tol=1e-11)
