"""S(q) on lattices of any shape: layers, columns, chains and more planes than a launch dimension
holds, on both ways the sums are taken, and a change of the replica count that changes the way.

The reference is the direct sum in FP64.  Phases are products of up to four table entries instead of
one exponential: 5 roundings per term of a sum of N terms of size 1, so |F|^2 <= N^2 is off by at most
about 2e-15 N^2."""
import math

import numpy as np
import pytest

from espins_amd import lattice as Lt

pytestmark = pytest.mark.gpu


def model(kind, Ls):
    nb = len(Lt.BASIS[kind])
    bf, rows, N = np.array(Lt.BASIS[kind], float), {"J": Lt.shell_rows(kind, [1.0])}, math.prod(Ls) * nb
    m = Lt.Model(kind, Ls, nb, bf, np.ones(N), Lt.build_table(nb, bf, np.ones(nb), Ls, rows["J"], 1), rows=rows)
    x2, x1, x0 = np.meshgrid(*[np.arange(n) for n in Ls[::-1]], indexing="ij")
    cells = np.stack([x0, x1, x2], -1).reshape(-1, 1, 3)
    return m, (cells + bf[None]).reshape(-1, 3).astype(float)


def mesh(n, axes):
    t = np.arange(n) / max(n - 1, 1) * 2 * math.pi
    q = np.zeros((n * n, 3))
    q[:, axes[0]], q[:, axes[1]] = np.repeat(t, n), np.tile(t, n)
    return q


def direct(s, pos, q, polar):
    e = np.exp(1j * (q @ pos.T))
    q2 = (q * q).sum(1)
    ok = q2 > 0
    out = np.zeros((len(s), 3, len(q)))
    for r in range(len(s)):
        F = e @ s[r]
        F = F[ok] - (F[ok] * q[ok]).sum(1)[:, None] * q[ok] / q2[ok][:, None]
        f2 = (np.abs(F) ** 2).sum(1)
        nsf2 = (F @ polar / np.linalg.norm(polar)).real ** 2
        out[r][:, ok] = f2, f2 - nsf2, nsf2
    return out


def measure(eng, R, q):
    eng.run(1, measure=True, exchange=False, seed=2 + R)
    got, n = eng.obs(16, (R, 3, len(q)))
    assert n == 1
    return got, eng.spins()


@pytest.mark.parametrize("kind,Ls", [("sc", (64, 64, 1)), ("fcc", (24, 24, 1)), ("sc", (1, 1, 66000)), ("sc", (2, 2, 300)),
                                     ("sc", (1, 700, 1)), ("bcc", (900, 1, 1)), ("fcc", (40, 3, 7)), ("sc", (8, 8, 33))])
@pytest.mark.parametrize("qk,R", [("xz", 1), ("yx", 6)])
def test_shapes(kind, Ls, qk, R):
    from espins_amd.engine import Engine
    print(kind, Ls, qk, R, flush=True)
    m, pos = model(kind, Ls)
    q = mesh(2 if m.N > 50000 else 9, ["xyz".index(a) for a in qk])
    polar = np.array([0.2, -0.5, 0.7])
    with Engine(0) as eng:
        eng.set_path(1)
        eng.set_model(m)
        eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 4))
        eng.set_sfactor(q, pos, polar, every=1)
        got, s = measure(eng, R, q)
    # (q.r of the longest chain is 2 pi 66000, whose own rounding is 6e-11)
    assert np.allclose(got, direct(s, pos, q, polar), rtol=1e-11, atol=(1e-13 + 1e-16 * pos.max()) * m.N ** 2)


def test_replica_count_changes_the_way():
    """With one replica the chain of a wave decides, with 64 the whole work."""
    from espins_amd.engine import Engine
    m, pos = model("sc", (40, 8, 8))
    q, polar = mesh(27, (0, 2)), np.array([0.2, -0.5, 0.7])
    with Engine(0) as eng:
        eng.set_path(1)
        eng.set_model(m)
        eng.set_sfactor(q, pos, polar, every=1)
        for R in (1, 64, 1):
            eng.set_replicas(np.linspace(0.5, 2.0, R), Lt.random_spins(m.N, R, 4))
            got, s = measure(eng, R, q)
            assert np.allclose(got, direct(s, pos, q, polar), rtol=1e-11, atol=1e-13 * m.N ** 2)
