"""Order parameter, staggered moment and P(m) of cells of 1 to 9 atoms, which are read four at a time
and then what is left, against the oracle's on the configuration measured."""
import numpy as np
import pytest

from espins_amd import lattice as Lt
from oracle import obs_oracle as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_cells_of_every_size(nb):
    from espins_amd.engine import Engine
    print(nb, flush=True)
    ncell, R = 300, 3                                     # rings of cells, atom by atom
    N, cell = ncell * nb, np.repeat(np.arange(ncell), nb)
    atom = np.tile(np.arange(nb), ncell)
    nbr = np.array([(cell + s) % ncell * nb + atom + 1 for s in (1, -1)], np.int32)
    m = Lt.Model("ring", (ncell, 1, 1), nb, np.zeros((nb, 3)), np.ones(N),
                 Lt.Table(2, np.full(N, 2, np.int32), nbr, np.ones((2, N))))
    rng = np.random.default_rng(nb)
    axes, coeff = rng.normal(size=(nb, 3)), rng.choice([-1.0, 1.0], nb)
    with Engine(0) as eng:
        eng.set_model(m)
        eng.set_replicas([0.5, 1.0, 2.0], Lt.random_spins(N, R, 5))
        eng.set_orderparam(axes)
        eng.set_staggered(coeff)
        nfreq = eng.set_pm(True)
        eng.run(1, measure=True, exchange=False, seed=7)
        s = eng.spins()
        op, _ = eng.obs(1, (R, 3))
        sm, _ = eng.obs(2, (R, 3))
        pm, _ = eng.obs(4, (R, 3, nfreq))
    for r in range(R):
        a, b = B.orderparam(s[r], nb, axes), B.staggered(s[r], nb, coeff)
        # sums of N terms of size 1, divided by the cells: N eps
        np.testing.assert_allclose(op[r], [abs(a), a * a, a ** 4], rtol=0, atol=1e-12 * nb ** 4)
        np.testing.assert_allclose(sm[r], [b, b * b, b ** 4], rtol=0, atol=1e-12 * nb ** 4)
        assert np.array_equal(pm[r], B.pm_counts(s[r], nb, m.mag[:nb], axes=axes, coeff=coeff))
