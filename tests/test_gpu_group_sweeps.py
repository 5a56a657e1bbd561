"""DIC / DILU and Gauss-Seidel sweeps run by a group of workgroups, on one XCD
(small levels) and on all (larger ones), against the oracle, bit for bit: the sizes where the packed tables and the
runs of a level can go wrong (rows not a multiple of a wavefront's, levels of
one row, levels of several items, rows longer than the packed entries and
than one overflow chunk), and values changed after the tables were made."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


def _rng(n, seed):
    return np.random.default_rng(seed).uniform(-1, 1, n)


def _fans(n, hubs, seed):
    """A ring of n cells with `hubs` cells joined to many others: rows of
    2 .. n entries, owner-sorted faces, diagonally dominant."""
    g = np.random.default_rng(seed)
    pairs = {(i, i + 1) for i in range(n - 1)}
    for h in range(hubs):
        c = int(g.integers(0, n))
        for o in g.choice(n, size=int(g.integers(7, min(n, 150))), replace=False):
            if o != c:
                pairs.add((min(c, int(o)), max(c, int(o))))
    l, u = np.array(sorted(pairs), np.int64).T
    up, lo = -g.uniform(0.1, 1, l.size), -g.uniform(0.1, 1, l.size)
    d = np.ones(n)
    np.add.at(d, l, np.abs(up))
    np.add.at(d, u, np.abs(lo))
    return meshgen.LduSystem(n, l.copy(), u.copy(), lo, d, up, _rng(n, seed + 1), False)


def _system(name):
    kind, dims = name
    if kind == "fans":
        return _fans(*dims)
    p = {"poisson": (meshgen.POISSON_LOGUNIF, -3.0, 0.0, 1e-6), "convdiff": (meshgen.CONVDIFF, 5.0, 0.0, 1e-3)}[kind]
    return meshgen.box_system(*dims, *p, 77)


SYSTEMS = [("poisson", (1, 1, 2)), ("poisson", (1, 1, 70)), ("convdiff", (17, 19, 23)), ("poisson", (40, 41, 39)),
           ("convdiff", (64, 63, 65)), ("poisson", (90, 91, 89)), ("fans", (9, 1, 3)), ("fans", (700, 40, 4)), ("fans", (3000, 200, 5))]


@pytest.mark.parametrize("name", SYSTEMS, ids=str)
def test_dilu_and_dic(oracle, name):
    s = _system(name)
    kind = "DIC" if s.symmetric else "DILU"
    A = hip.LduMatrix.from_system(s)
    P = hip.Precond(A, kind)
    for seed in (3, 4, 5, 6):
        r = _rng(s.n, seed)
        assert np.array_equal(P.apply(r), oracle.matrix(s).precond(kind, r)[0])


@pytest.mark.parametrize("name", SYSTEMS, ids=str)
def test_gauss_seidel(oracle, name):
    s = _system(name)
    A = hip.LduMatrix.from_system(s)
    x0 = _rng(s.n, 5)
    S = hip.Smoother("GS")
    for sweeps in (1, 4, 11):
        assert np.array_equal(S.smooth(A, x0, s.b, sweeps), oracle.matrix(s).smooth("GS", x0, s.b, sweeps))


def test_gauss_seidel_on_coarse_levels(oracle):
    # agglomerated levels: rows of 10 .. 40 entries, 8 and 4 lanes a row
    s = _system(("poisson", (30, 31, 29)))
    G = oracle.matrix(s).agglomerate(np.abs(s.upper), n_coarsest=30)
    for lv in G:
        c = meshgen.LduSystem(lv["n"], lv["l"], lv["u"], None, lv["diag"], lv["upper"], _rng(lv["n"], 6), True)
        A = hip.LduMatrix.from_system(c)
        x0 = _rng(c.n, 7)
        assert np.array_equal(hip.Smoother("GS").smooth(A, x0, c.b, 3), oracle.matrix(c).smooth("GS", x0, c.b, 3))


def test_new_coefficients(oracle):
    s = _system(("convdiff", (17, 19, 23)))
    A = hip.LduMatrix.from_system(s)
    S = hip.Smoother("GS")
    x0 = _rng(s.n, 8)
    S.smooth(A, x0, s.b, 2)
    hip.Precond(A, "DILU").apply(s.b)
    t = meshgen.LduSystem(s.n, s.l, s.u, s.lower * 0.7, s.diag * 1.1, s.upper * 0.9, s.b, False)
    A.set_coeffs(t.diag, t.upper, t.lower)
    assert np.array_equal(S.smooth(A, x0, t.b, 2), oracle.matrix(t).smooth("GS", x0, t.b, 2))
    assert np.array_equal(hip.Precond(A, "DILU").apply(t.b), oracle.matrix(t).precond("DILU", t.b)[0])
