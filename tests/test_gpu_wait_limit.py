"""A wait between workgroups that gives up ends the call in an error, leaves no
launch waiting, and the next call answers right.  The wait is made to give up
by a limit of no polls, so every kernel still runs to its end."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_polls():
    def calls(f):
        hip.set_wait_limit(0)
        try:
            with pytest.raises(hip.UnapHipError, match="waited too long"):
                f()
        finally:
            hip.set_wait_limit()
    return calls


# levels small enough for the workgroups of one XCD, and for those of all
@pytest.mark.parametrize("dims", [(40, 41, 39), (90, 91, 89)], ids=str)
def test_sweeps(oracle, no_polls, dims):
    s = meshgen.box_system(*dims, meshgen.CONVDIFF, 5.0, 0.0, 1e-3, 5)
    A = hip.LduMatrix.from_system(s)
    x0 = np.random.default_rng(6).uniform(-1, 1, s.n)
    S, P, O = hip.Smoother("GS"), hip.Precond(A, "DILU"), oracle.matrix(s)
    for _ in range(2):
        no_polls(lambda: S.smooth(A, x0, s.b, 4))
        assert np.array_equal(S.smooth(A, x0, s.b, 4), O.smooth("GS", x0, s.b, 4))
        no_polls(lambda: P.apply(s.b))
        assert np.array_equal(P.apply(s.b), O.precond("DILU", s.b)[0])


@pytest.mark.parametrize("graphs", [True, False])
def test_solves(oracle, no_polls, graphs):
    s = meshgen.box_system(40, 41, 39, meshgen.POISSON_LOGUNIF, -3.0, 0.0, 1e-6, 5)
    A = hip.LduMatrix.from_system(s)
    hip.set_graph_replay(graphs)
    try:
        for pre, amg in (("DIC", None), ("AMG", hip.amg_params(smoother=1, n_cells_coarsest=100, n_vcycles=1))):
            S = hip.Solver("PCG", hip.Precond(A, pre, amg=amg), rel_tol=1e-8, max_iter=300)
            x, p = S.solve(A, s.b)
            assert p["converged"]
            for _ in range(2):
                no_polls(lambda: S.solve(A, s.b))
                y, q = S.solve(A, s.b)
                assert np.array_equal(x, y) and p["nIterations"] == q["nIterations"]
    finally:
        hip.set_graph_replay(True)


def test_teams(no_polls):
    systems = [meshgen.box_system(33, 31, 29, meshgen.POISSON_LOGUNIF, -3.0, 0.0, 1e-6, 1),
               meshgen.box_system(30, 27, 35, meshgen.CONVDIFF, 5.0, 0.0, 1e-3, 2)]
    systems += [meshgen.box_system(8, 8, 8, meshgen.POISSON_CONST, 0.0, 0.0, 1e-2, i) for i in range(20)]
    B = hip.Batch(systems, ["PCG" if s.symmetric else "PBiCGStab" for s in systems])
    B.set_config(1024, 1, 128)
    b = np.concatenate([s.b for s in systems])
    x, p = B.solve(b)
    assert all(q["converged"] for q in p)
    for _ in range(2):
        no_polls(lambda: B.solve(b))
        y, q = B.solve(b)
        assert np.array_equal(x, y) and [v["nIterations"] for v in p] == [v["nIterations"] for v in q]


def test_refused_limits():
    for polls in (-1, (1 << 23) + 1):
        with pytest.raises(hip.UnapHipError):
            hip.set_wait_limit(polls)
