"""S(q) on lattice positions, summed axis by axis over the distinct pairs (q.A0, q.A1), against the
oracle's direct sum: a mesh whose points share pairs, points that share none (more pairs than one
wave's lanes), a single point, odd and even edges, partial replica groups.

The phases are products of three table entries instead of one exponential: 4 roundings per term of
a sum of N terms of size 1, so |F|^2 <= N^2 is off by at most about 1e-15 N^2."""
import math

import numpy as np
import pytest

from espins_amd import lattice as Lt
from oracle import obs_oracle as B

pytestmark = pytest.mark.gpu


def q_points(kind, n):
    rng = np.random.default_rng(n)
    if kind == "mesh":
        ij = np.array([(i, j) for i in range(n) for j in range(n)], float) / max(n - 1, 1)
        return 2 * math.pi * (ij[:, :1] * [1.0, 0, 0] + ij[:, 1:] * [0, 0, 1.0])
    return rng.uniform(-7.0, 7.0, size=(n, 3))


@pytest.mark.parametrize("kind,L,R", [("sc", 5, 1), ("sc", 8, 6), ("fcc", 5, 5), ("bcc", 6, 4)])
@pytest.mark.parametrize("qk,n", [("mesh", 1), ("mesh", 9), ("random", 70)])
def test_sfactor_by_planes(kind, L, R, qk, n):
    from espins_amd.engine import Engine
    print(kind, L, R, qk, n, flush=True)
    m = Lt.cubic_model(kind, L, J=(1.0,))
    pos, q, polar = Lt.site_positions(kind, L), q_points(qk, n), np.array([0.2, -0.5, 0.7])
    with Engine(0) as eng:
        eng.set_path(1)
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 4))
        eng.set_sfactor(q, pos, polar, every=1)
        eng.run(1, measure=True, exchange=False, seed=2)
        got, count = eng.obs(16, (R, 3, len(q)))
        s = eng.spins()
    want = np.stack([B.sfactor(s[r], pos, q, polar) for r in range(R)])
    assert count == 1
    assert np.allclose(got, want, rtol=1e-11, atol=1e-13 * m.N ** 2)


@pytest.mark.parametrize("bad", [[0], [3], [0, 5, 6]])
def test_points_that_are_not_numbers(bad):
    """A q-point that is not a number spoils its own S(q) only."""
    from espins_amd.engine import Engine
    m = Lt.cubic_model("sc", 6, J=(1.0,))
    pos, q, polar = Lt.site_positions("sc", 6), q_points("random", 9), np.array([0.2, -0.5, 0.7])
    q[bad, 0] = [np.nan, np.inf, np.nan][:len(bad)]
    with Engine(0) as eng:
        eng.set_path(1)
        eng.set_model(m)
        eng.set_replicas([0.5, 1.0], Lt.random_spins(m.N, 2, 4))
        eng.set_sfactor(q, pos, polar, every=1)
        eng.run(1, measure=True, exchange=False, seed=2)
        got, _ = eng.obs(16, (2, 3, len(q)))
        s = eng.spins()
    good = np.setdiff1d(np.arange(len(q)), bad)
    want = np.stack([B.sfactor(s[r], pos, q[good], polar) for r in range(2)])
    assert np.allclose(got[:, :, good], want, rtol=1e-11, atol=1e-13 * m.N ** 2)
    assert np.isnan(got[:, 0, bad]).all()
