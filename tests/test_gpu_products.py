"""Products of the module API that one launch forms and writes to the host
(energyprod_edge2d, massprod_edge2d, dotprod_*) on both sides of one workgroup
and up to the most workgroups, twice in a row, and the M-orthonormalisation's
two launches per reflection at its edges (one vector, more than the 48 whose
coefficients fit the LDS, one to 64 partial sums per vector, a zero vector, a
nearly dependent one), against the oracle.

Tolerances: a sum of n products rounds to a few eps (a tree of depth log n
over sums of at most n / 2^18 terms) of the product of the norms: 1e-14 of
it; the orthonormalisation 1e-12 as the drivers' sizes."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rnd(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("nx,ny", [(2, 2), (64, 64), (66, 64), (30, 258), (640, 512)])
def test_products(nx, ny):
    import maxwell_amd as M
    print("products %d x %d" % (nx, ny), flush=True)
    rng = np.random.default_rng(nx + ny)
    eta, kx, ky = 1.0 / rng.uniform(1.0, 9.0, size=(ny, nx)), 0.6, -2.9
    G, g = M.Grid(eta, kx, ky, hx=1 / nx, hy=0.9 / ny), O.Grid2D(eta, 1 / nx, 0.9 / ny, kx, ky)
    x, y, a, b = rnd(rng, g.nedge), rnd(rng, g.nedge), rnd(rng, g.nnode), rnd(rng, g.nnode)
    X, Y, A, B = M.Edge(G, x), M.Edge(G, y), M.Node(G, a), M.Node(G, b)
    al, be = 0.3 - 1.0j, 0.7 + 0.2j
    tx, mx = O.addeval(g, al, be, x), O.addeval(g, 0.0, 1.0, x)
    n = np.linalg.norm
    for _ in range(2):
        e = M.lib.energyprod_edge2d(M.Cplx.of(al), M.Cplx.of(be), X.h, Y.h).value()
        assert abs(e - np.conj(np.vdot(y, tx))) <= 1e-14 * n(y) * n(tx)
        m = M.lib.massprod_edge2d(X.h, Y.h).value()
        assert abs(m - np.conj(np.vdot(y, mx))) <= 1e-14 * n(y) * n(mx)
        d = M.lib.dotprod_edge2d(X.h, Y.h).value()
        assert abs(d - np.vdot(x, y)) <= 1e-14 * n(x) * n(y)
        d = M.lib.dotprod_node2d(A.h, B.h).value()
        assert abs(d - np.vdot(a, b)) <= 1e-14 * n(a) * n(b)


@pytest.mark.parametrize("nx,ny,k,special", [(16, 16, 1, None), (16, 16, 49, None), (34, 32, 20, "zero"),
                                             (16, 48, 9, "near"), (6, 4, 12, None), (258, 256, 3, None),
                                             (5, 7, 4, None)])
def test_orthonormalize_edges(nx, ny, k, special):
    import maxwell_amd as M
    print("orthonormalize %d x %d, %d vectors, %s" % (nx, ny, k, special), flush=True)
    rng = np.random.default_rng(nx + k)
    eta, kx, ky = np.ones((ny, nx)), -0.8, 1.7
    hx, hy = 1.0 / nx, 0.8 / ny
    G, g = M.Grid(eta, kx, ky, hx=hx, hy=hy), O.Grid2D(eta, hx, hy, kx, ky)
    X = rnd(rng, k, 2 * nx * ny)
    if special == "zero":
        X[k // 2] = 0
    if special == "near":
        X[k - 1] = X[0] + 1e-3 * X[k - 1]
    edges = [M.Edge(G, v) for v in X]
    tau = (M.Cplx * k)()
    M.lib.orthonormalize_edge2d(k, (C.c_void_p * k)(*[e.h for e in edges]), tau, None)
    out = np.array([e.get() for e in edges])
    ref, tref, _ = O.orthonormalize(g, X)
    # a nearly dependent vector: its remainder's rounding, a thousandfold
    tol = 1e-9 if special == "near" else 1e-12
    assert np.abs(out - ref).max() <= tol * np.abs(ref).max()
    assert np.abs(np.array([t.value() for t in tau]) - tref).max() <= tol * np.abs(tref).max()
    Mout = np.array([O.addeval(g, 0.0, 1.0, v) for v in out])
    assert np.abs(out.conj() @ Mout.T - np.eye(k)).max() <= 1e-12
