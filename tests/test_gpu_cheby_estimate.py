"""Chebyshev eigenvalue estimates of levels on which the ten CG steps meet a
zero residual before the tenth (a strong diagonal in FP32: w r underflows):
the estimate is formed from the steps that were made."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("off", [1e-2, 1e-4, 1e-8])
def test_strong_diagonal(off, precision):
    s = meshgen.config_system(4, 20)
    A = hip.LduMatrix(s.n, s.l, s.u, None, s.diag, s.upper * off)
    P = hip.Precond(A, "AMG", amg=hip.amg_params(smoother=2, n_cells_coarsest=50, n_vcycles=1, n_post_sweeps=4,
                                                  n_finest_sweeps=4, precision=precision, pair_steps=2,
                                                  cycle=hip.CYCLE_FIXED))
    x, p = hip.Solver("FCG", P, rel_tol=1e-8, max_iter=60).solve(A, s.b)
    r = s.b - s.diag * x
    np.add.at(r, s.l, -off * s.upper * x[s.u])
    np.add.at(r, s.u, -off * s.upper * x[s.l])
    assert p["converged"] and np.linalg.norm(r) <= 2e-8 * np.linalg.norm(s.b), p
