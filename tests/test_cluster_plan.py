"""Planning the clusters of blocks (host only): parts and sites of the plans against a direct count
from the bond tables, and the time that a model too large for clusters costs."""
import time

import numpy as np
import pytest

from espins_amd import lattice as Lt
from espins_amd.engine import plan_clusters, plan_model


def most_sites(m, k):
    """Sites of the largest of k parts of consecutive sites, with the foreign sites its bonds reach."""
    part = np.arange(m.N) * k // m.N
    t = m.J
    bond = np.arange(t.z)[:, None] < t.cnt
    i, j = np.tile(np.arange(m.N), (t.z, 1))[bond], t.nbr.reshape(t.z, m.N)[bond] - 1
    out = part[i] != part[j]
    halo = np.unique(part[i][out].astype(np.int64) * m.N + j[out]) // m.N
    return int((np.bincount(part, minlength=k) + np.bincount(halo, minlength=k)).max())


@pytest.mark.parametrize("kind,L,J,R,fits", [("fcc", 16, (1.0, 0.1), 64, True), ("sc", 14, (1.0,), 32, True),
                                             ("sc", 20, (1.0,), 24, True), ("bcc", 9, (1.0, -0.2), 64, True),
                                             ("sc", 64, (1.0,), 1, True), ("sc", 48, (1.0,), 8, False),
                                             ("sc", 6, (1.0,), 8, False)])
def test_plans(kind, L, J, R, fits):
    m = Lt.cubic_model_fast(kind, L, J=J)
    p = plan_clusters(m, R)
    # a CU for every part, a wave's sites of each colour in it
    parts = min(256 // R, m.N // plan_model(m)[0] // 64) if fits else 0
    assert p["parts"] == parts and p["lds"] <= 160 * 1024
    assert p["sites"] == (most_sites(m, parts) if parts else 0)


@pytest.mark.parametrize("L,R", [(80, 2), (100, 1)])
def test_a_model_too_large_is_declined_at_once(L, R):
    """Parts of a large lattice never fit: their halo is two layers.  Seeing that must cost no more
    than the model's own preparation (a try for every smaller number of parts cost up to 26 s)."""
    m = Lt.cubic_model_fast("sc", L, J=(1.0,))
    t0 = time.process_time()
    plan_model(m)
    t1 = time.process_time()
    assert plan_clusters(m, R)["parts"] == 0
    t2 = time.process_time()
    assert t2 - t1 < 2.0 * (t1 - t0) + 0.2
