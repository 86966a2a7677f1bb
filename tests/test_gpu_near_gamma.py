"""LOBPCG next to the Gamma point on a fine grid: the lowest eigenvalue is small
against the Ritz values of the rounding noise that the basis comes to hold, so
its residual only falls below the tolerance if the small eigenproblems keep the
small components of their vectors.  Several start blocks at one k all converge
to the same eigenvalues."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def test_lobpcg_near_gamma_converges_from_every_start():
    import maxwell_amd as M
    k = 0.12038850145632063
    S = M.Solver(O.rod_eta(512), n0=4, levels=7, precision=1, block=12, max_problems=32, method=M.MX_METHOD_LOBPCG)
    r = S.solve([k] * 32, [k] * 32, neig=10, tol=1e-8, maxit=60, seed=5)
    S.close()
    assert r["converged"].all(), (r["iters"], r["relres"][:, 0])
    lam = r["lam"][:, :10]
    # a residual of 1e-8 bounds a Ritz value's relative error by its square
    # over the gaps: far below 1e-9
    assert np.abs(lam - lam[0]).max() <= 1e-9 * lam[0, -1]
