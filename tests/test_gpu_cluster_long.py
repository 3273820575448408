"""Runs on clusters of blocks whose steps or rounds are longer than one launch (2^18 colour phases):
launches end between the steps of a round and within a step, and the measurements, exchanges and
counts are those of the launch-per-colour path."""
import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu
PHASES = 1 << 18


@pytest.mark.parametrize("rounds,steps,M,exchange", [(2, 2, 33000, True), (1, 3, 12000, False), (3, 2, 12000, True)])
def test_steps_longer_than_a_launch(rounds, steps, M, exchange):
    from espins_amd.engine import Engine
    print(rounds, steps, M, exchange, flush=True)
    m = Lt.cubic_model("fcc", 6, J=(1.0, 0.2))
    R = 4
    out = []
    for path in (0, 1):
        with Engine(0) as eng:
            eng.set_path(path)
            eng.set_model(m)
            eng.set_replicas(np.linspace(0.6, 2.0, R), Lt.random_spins(m.N, R, 5))
            eng.set_trace(8)
            eng.run(rounds, steps_per_round=steps, steps_measure=M, measure=True, exchange=exchange, seed=12)
            ncol, _ = eng.coloring()
            if path == 0:
                most = PHASES // ncol            # sweeps of a launch
                info = eng.cluster_info()
                assert info["sweeps"] == rounds * steps * M
                n = rounds * steps
                assert info["launches"] == (n * -(-M // most) if M > most else -(-n // (most // M)))
            out.append((eng.stats(), eng.spins(), eng.pt_map(), eng.trace(), eng.energy_get()))
    a, b = out
    assert a[0]["nmeas"] == b[0]["nmeas"] == rounds * steps
    assert np.array_equal(a[0]["rejected"], b[0]["rejected"])
    assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
    np.testing.assert_allclose(a[1], b[1], rtol=0, atol=1e-13)
    # running energies: 1e5 sweeps of 864 differences, each rounded to 1e-16 of their size
    np.testing.assert_allclose(a[3], b[3], rtol=1e-9, atol=1e-7)
    np.testing.assert_allclose(a[0]["e_run"], a[4], rtol=1e-9, atol=1e-7)
