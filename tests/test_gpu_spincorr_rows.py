"""Spin correlations over shells of 1 to 8 partner rows, which are read three at a time and then one by
one, for one kind and several, against the oracle's on the configuration measured."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from oracle import obs_oracle as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [1, 2, 3])
@pytest.mark.parametrize("sizes", [(1,), (2, 5), (3, 4, 1), (8, 7, 6)])
def test_shells_of_every_size(sizes, kinds):
    from espins_amd.engine import Engine
    print(sizes, kinds, flush=True)
    N, R, ns = 402, 3, len(sizes)      # a ring; each row of a shell is one step to both sides
    i = np.arange(N)
    nbr, cnt = np.zeros((ns, 2 * max(sizes), N), np.int32), np.zeros((ns, N), np.int32)
    at = 1
    for k, n in enumerate(sizes):
        for s in range(n):
            nbr[k, 2 * s], nbr[k, 2 * s + 1] = (i + at) % N + 1, (i - at) % N + 1
            at += 1
        cnt[k] = 2 * n
    m = Lt.Model("ring", (N, 1, 1), 1, np.zeros((1, 3)), np.ones(N),
                 Lt.Table(2, np.full(N, 2, np.int32), np.array([(i + 1) % N + 1, (i - 1) % N + 1], np.int32), np.ones((2, N))))
    species = (i % kinds).astype(np.int32)
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas([0.5, 1.0, 2.0], Lt.random_spins(N, R, 5))
        eng.set_spincorr(species, cnt, nbr)
        eng.run(1, measure=True, exchange=False, seed=7)
        s = eng.spins()
        sc, _ = eng.obs(8, (R, 3, ns, kinds, kinds))
    for r in range(R):
        t, ta = B.spincorr(s[r], species, cnt, nbr, m.mag, kinds)
        # sums of n = 2 rows N terms of at most 1 in another order: n eps of the sum of their sizes
        for got, want in ((sc[r, 0], t), (sc[r, 1], np.abs(t)), (sc[r, 2], ta)):
            np.testing.assert_allclose(got, want, rtol=0, atol=2 * max(sizes) * N * 2.3e-16 * N)
