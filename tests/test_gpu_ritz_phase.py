"""A pair that has converged is carried through the Ritz step unchanged: its
coefficient is real and 1 to the last bit, so that its vector is not rounded
anew in every step.  Next to the Gamma point on a fine grid that rounding is
what the residual consists of (eps |K| / lambda, about 1e-8 on 512 x 512 at
|k| = 0.12): a vector multiplied by a complex phase every step came to lie above
the tolerance again and again, and the solve never ended.

Bounds of the kernel's test.  M = 1 and K = diag(d) + E with |E_ij| <= 1e-10 and
gaps of at least 13: every rotation's angle is below 1e-11, whose square is lost
against 1, so the diagonal's real parts are products of ones.  Its imaginary
parts and what the other entries differ from first-order perturbation theory,
-E_ij / (d_i - d_j), are sums of at most m products of two angles (32 x 1e-22),
and the rounding of the quotients (1e-11 eps cond, 1e-25)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import test_gpu_ritz as R
from test_gpu_ritz import lib  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 5, 12, 17, 32])
def test_converged_pairs_keep_their_vectors(lib, m):  # noqa: F811
    print("ritz, %d converged pairs" % m, flush=True)
    rng = np.random.default_rng(m)
    d = 0.0145 + 13.0 * np.arange(m)
    E = 1e-10 * np.triu(np.exp(2j * np.pi * rng.random((m, m))), 1)
    E = E + E.conj().T
    Cm, lam, st = R.run(lib, m, 0, [R.pack(np.diag(d) + E, np.eye(m) + 0j, m, 4.0)], [[]], 4.0, 1e-13)
    assert st[0] == 0
    c = Cm[0]
    assert (np.diag(c).real == 1.0).all()
    gap = d[None, :] - d[:, None] + np.eye(m)
    first = np.where(np.eye(m) > 0, 1.0, E / gap)
    assert np.abs(c - first).max() <= 1e-20
    assert np.abs(lam[0][:m] - 1.0 - d).max() <= 1e-12


@pytest.mark.parametrize("k,least", [(0.085, 32), (0.08, 4)])
def test_pinvit_near_gamma(k, least):
    """At 0.085 rounding leaves the lowest pair's residual just below the
    tolerance in every start block; at 0.08 in about half of them (90 of 160
    with the eigenproblems solved one rotation at a time on the host), and in
    none where it is rounded anew in every step."""
    import maxwell_amd as M
    S = M.Solver(O.rod_eta(512), n0=4, levels=7, precision=1, block=12, max_problems=32)
    r = S.solve([k] * 32, [k] * 32, neig=10, tol=1e-8, maxit=120, seed=5)
    S.close()
    assert r["converged"].sum() >= least, (r["iters"], r["relres"][:, 0])
    lam = r["lam"][r["converged"], :10]
    # a residual of 1e-8 bounds a Ritz value's relative error by its square over the gaps
    assert np.abs(lam - lam[0]).max() <= 1e-9 * lam[0, -1]
