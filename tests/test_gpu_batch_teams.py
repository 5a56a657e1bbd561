"""Batched systems solved by teams of workgroups: the same bits whatever the
team's size (eight workgroups in a batch of few systems, four in a batch of
many), and true residuals within the tolerance."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


def _diagonal(n):
    e = np.zeros(0, np.int64)
    rng = np.random.default_rng(n)
    return meshgen.LduSystem(n, e, e.copy(), None, 1.0 + rng.random(n), np.zeros(0), rng.uniform(-1, 1, n), True)


def _solve(systems, kinds):
    B = hip.Batch(systems, kinds)
    B.set_config(1024, 2, 256)
    x, p = B.solve(np.concatenate([s.b for s in systems]), rel_tol=1e-8, max_iter=1000)
    return [x[B.cell_off[i]:B.cell_off[i + 1]] for i in range(len(systems))], p


def test_team_sizes(oracle):
    # randomly numbered boxes of few wide levels; rows not a multiple of 64; one level only
    big = [meshgen.box_system(33, 31, 29, meshgen.POISSON_LOGUNIF, -3.0, 0.0, 1e-6, 1),
           meshgen.box_system(30, 27, 35, meshgen.CONVDIFF, 5.0, 0.0, 1e-3, 2), _diagonal(5001)]
    kinds = ["PCG", "PBiCGStab", "PCG"]
    small = [meshgen.box_system(8, 8, 8 + i % 3, meshgen.POISSON_CONST, 0.0, 0.0, 1e-2, i) for i in range(200)]
    x8, p8 = _solve(big, kinds)
    x4, p4 = _solve(big + small, kinds + ["PCG"] * len(small))
    for i, s in enumerate(big):
        assert np.array_equal(x8[i], x4[i]) and p8[i]["nIterations"] == p4[i]["nIterations"], i
    for i, s in enumerate(big + small):
        r = s.b - oracle.matrix(s).spmv(x4[i])
        assert p4[i]["converged"] and np.linalg.norm(r) <= 2e-8 * np.linalg.norm(s.b), i
