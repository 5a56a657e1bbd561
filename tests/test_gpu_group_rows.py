"""Sweeps in one launch on rows longer than the packed entries: more than six
entries a side (DIC / DILU, FP64 and FP32), rows of two, three and more overflow
chunks at 2, 4 and 8 lanes a row (Gauss-Seidel), by the workgroups of one XCD
and of all, bit for bit.  The systems are layers of cells joined to random cells
of earlier layers, so that they have few levels, and each test asks for the
route it means to take."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


def _layers(layers, width, most, hubs, seed, symmetric=False):
    """`layers` layers of about `width` cells, a cell joined to 0 .. `most`
    cells of earlier layers and `hubs` cells a layer to up to 150."""
    g = np.random.default_rng(seed)
    start = np.concatenate([[0], np.cumsum(g.integers(width - width // 7, width + 1, layers))])
    n = int(start[-1])
    l, u = [], []
    for k in range(1, layers):
        for c in range(start[k], start[k + 1]):
            many = 150 if c < start[k] + hubs else most
            for o in g.choice(start[k], size=min(int(start[k]), int(g.integers(0, many + 1))), replace=False):
                l.append(int(o))
                u.append(c)
    l, u = np.array(l, np.int64), np.array(u, np.int64)
    at = np.lexsort((u, l))
    l, u = l[at], u[at]
    up = -g.uniform(0.1, 1, l.size)
    lo = up.copy() if symmetric else -g.uniform(0.1, 1, l.size)
    d = np.full(n, 0.5)
    np.add.at(d, l, np.abs(up))
    np.add.at(d, u, np.abs(lo))
    return meshgen.LduSystem(n, l, u, None if symmetric else lo, d, up, g.uniform(-1, 1, n), symmetric)


def _rows(s):
    lower, upper = np.bincount(s.u, minlength=s.n), np.bincount(s.l, minlength=s.n)
    return lower, upper


# name -> (layers, width, most, hubs, seed); GS lanes a row 2 / 4 / 8; XCDs of (LU, GS)
SYSTEMS = {
    "two lanes": ((7, 400, 5, 6, 1), 2, 1, 1),
    "four lanes": ((9, 300, 9, 3, 2), 4, 1, 1),
    "eight lanes": ((6, 250, 24, 9, 3), 8, 1, 1),
    "two lanes, wide": ((5, 16000, 5, 20, 4), 2, 8, 8),
    "four lanes, wide": ((4, 11000, 11, 20, 5), 4, 8, 8),
    "eight lanes, wide": ((4, 9000, 20, 20, 6), 8, 8, 8),
}


def _system(name, symmetric=False):
    args, lanes, lu, gs = SYSTEMS[name]
    s = _layers(*args, symmetric=symmetric)
    lower, upper = _rows(s)
    assert lower.max() > 12 and upper.max() > 12  # past the six packed entries of either side
    assert (lower + upper).max() > 3 * 4 * lanes  # past two overflow chunks
    average = (lower + upper).mean()
    assert average <= 7.0 if lanes == 2 else (7.0 < average <= 12.5 if lanes == 4 else average > 12.5)
    return s, lu, gs


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("name", SYSTEMS)
def test_dilu_and_dic(oracle, name, symmetric):
    s, lu, _ = _system(name, symmetric)
    A = hip.LduMatrix.from_system(s)
    kind = "DIC" if symmetric else "DILU"
    assert hip.sweep_xcds(A, "DIC") == lu
    P = hip.Precond(A, kind)
    for seed in (1, 2):
        r = np.random.default_rng(seed).uniform(-1, 1, s.n)
        assert np.array_equal(P.apply(r), oracle.matrix(s).precond(kind, r)[0])


@pytest.mark.parametrize("name", SYSTEMS)
def test_gauss_seidel(oracle, name):
    s, _, gs = _system(name)
    A = hip.LduMatrix.from_system(s)
    assert hip.sweep_xcds(A, "GS") == gs
    x0 = np.random.default_rng(3).uniform(-1, 1, s.n)
    for sweeps in (1, 3):
        assert np.array_equal(hip.Smoother("GS").smooth(A, x0, s.b, sweeps),
                              oracle.matrix(s).smooth("GS", x0, s.b, sweeps))


def _dilu32(s, rD, r):
    """The FP32 sweeps row by row: w = rD r, then (rD coefficient) w subtracted
    in face order; backward from the last face of the row."""
    f = np.float32
    lower = s.lower_or_upper().astype(f)
    upper = s.upper.astype(f)
    w = rD * r.astype(f)
    of_u = np.argsort(s.u, kind="stable")
    at_u = np.concatenate([[0], np.cumsum(np.bincount(s.u, minlength=s.n))])
    at_l = np.concatenate([[0], np.cumsum(np.bincount(s.l, minlength=s.n))])
    for c in range(s.n):
        acc = w[c]
        for e in of_u[at_u[c]:at_u[c + 1]]:
            acc = acc - (rD[c] * lower[e]) * w[s.l[e]]
        w[c] = acc
    for c in range(s.n - 1, -1, -1):
        acc = w[c]
        for e in range(at_l[c + 1] - 1, at_l[c] - 1, -1):
            acc = acc - (rD[c] * upper[e]) * w[s.u[e]]
        w[c] = acc
    return w


@pytest.mark.parametrize("name", ["two lanes", "eight lanes", "four lanes, wide"])
def test_fp32(name):
    s, _, _ = _system(name)
    A = hip.LduMatrix.from_system(s)
    P = hip.Precond(A, "DILU", precision=32)
    assert hip.sweep_xcds(A, "DIC", 32) == (8 if "wide" in name else 1)
    r = np.random.default_rng(5).uniform(-1, 1, s.n)
    assert np.array_equal(P.apply(r), _dilu32(s, P.rD().astype(np.float32), r).astype(np.float64))


def test_new_coefficients(oracle):
    # the overflow chunks and the entries past the packed ones follow new values
    s, _, _ = _system("four lanes")
    A = hip.LduMatrix.from_system(s)
    x0 = np.random.default_rng(6).uniform(-1, 1, s.n)
    S = hip.Smoother("GS")
    S.smooth(A, x0, s.b, 2)
    hip.Precond(A, "DILU").apply(s.b)
    t = meshgen.LduSystem(s.n, s.l, s.u, s.lower * 0.7, s.diag * 1.1, s.upper * 0.9, s.b, False)
    A.set_coeffs(t.diag, t.upper, t.lower)
    assert np.array_equal(S.smooth(A, x0, t.b, 2), oracle.matrix(t).smooth("GS", x0, t.b, 2))
    assert np.array_equal(hip.Precond(A, "DILU").apply(t.b), oracle.matrix(t).precond("DILU", t.b)[0])


def test_launched_level_by_level():
    # more levels than a launch holds
    n = 700
    l, u = np.arange(n - 1, dtype=np.int64), np.arange(1, n, dtype=np.int64)
    A = hip.LduMatrix.from_system(meshgen.LduSystem(n, l, u, None, np.full(n, 3.0), np.full(n - 1, -1.0), np.ones(n), True))
    assert hip.sweep_xcds(A, "GS") == 0 and hip.sweep_xcds(A, "DIC") == 0
