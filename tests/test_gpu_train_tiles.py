"""The training gradient against the oracle's FP64 gradient: one record, the edges of a wave's
records (16) and of a block's (128), and many blocks, the last one partial.

FP32 throughout: a unit's pre-activation sums 32 products and a gradient entry the records of a
block (then FP32 partial sums over blocks), so entries are off by about sqrt(32) 2^-24 per layer
through seven layers of forward and backward, 3e-6 of the largest entry; the bound is 1e-4 of it
(the oracle's mixture terms are FP64, the kernel's kappa and tilt FP32: 1e-6 relative on factors
that reach beta |G| ~ 50)."""
import numpy as np
import pytest

from espins_amd import learn as Ln
from oracle import learn_oracle as LO
from tests.test_learn_oracle import random_records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 128, 129, 512 * 32 + 33])
def test_gradient_at_tile_edges(n):
    from espins_amd.engine import Engine
    print("records", n, flush=True)
    recs = random_records(n, 40).astype(np.float32)
    w = Ln.init_weights(41, out_scale=0.4)
    with Engine() as eng:
        eng.learn_set_weights(w)
        eng.learn_put_records(recs)
        g, loss = eng.learn_grad()
        g2, loss2 = eng.learn_grad()
    L, go = LO.loss_and_grad(w.astype(np.float64), recs.astype(np.float64))
    assert loss == pytest.approx(L, rel=1e-5, abs=1e-5)
    np.testing.assert_allclose(g, go, rtol=0, atol=1e-4 * np.abs(go).max())
    assert np.array_equal(g, g2) and loss == loss2      # fixed order of every sum
