"""The one-workgroup coarsest solver against the oracle, bit for bit (reference
reduction order): coarsest levels on both sides of every thread-count line
(256, 512, 768, 1024 rows), a level of a handful of rows, and a level whose
rows are longer than a thread holds."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def reference_order():
    hip.set_reduction_order(hip.REDUCE_REFERENCE)
    yield
    hip.set_reduction_order(hip.REDUCE_TREE)


@pytest.mark.parametrize("edges,coarsest", [((9, 8, 7), 3), ((20, 19, 21), 150), ((20, 19, 21), 300), ((22, 23, 21), 400),
                                            ((23, 24, 25), 600), ((13, 12, 13), 800), ((13, 13, 14), 1000)])
def test_amg_pcg(oracle, edges, coarsest):
    s = meshgen.box_system(*edges, meshgen.POISSON_LOGUNIF, -3.0, 0.0, 1e-6, 31)
    A = hip.LduMatrix.from_system(s)
    P = hip.Precond(A, "AMG", amg=hip.amg_params(smoother=1, n_cells_coarsest=coarsest, n_vcycles=1))
    x, p = hip.Solver("PCG", P, rel_tol=1e-6, max_iter=30).solve(A, s.b)
    xo, po = oracle.matrix(s).solve("PCG", "AMG", s.b, rel_tol=1e-6, max_iter=30, mg=[1, coarsest, 1, 0, 2, 2])
    assert p["nIterations"] == po["nIterations"] and np.array_equal(p["history"], po["history"])
    assert np.array_equal(x, xo), P.amg_levels()
