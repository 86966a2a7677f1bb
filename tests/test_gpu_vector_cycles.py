"""The module API's V-cycles (fused passes, the coarse levels in one launch)
against the oracle's sweeps, residuals, restrictions and prolongations: every
level's right-hand side and solution."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import maxwell_amd
    return maxwell_amd


def arr(objs):
    return (C.c_void_p * len(objs))(*[o.h for o in objs])


def cycle(gs, node, l, b, x, nu, coarse, low):
    g = gs[l]
    sweep = O.gs_node if node else O.gs_edge
    if l == 0 and coarse:
        x = np.linalg.solve(O.dense_node(g, fixnull=True) if node else O.dense_edge(g, 1.0, 1.0), b)
    elif l == 0:
        for _ in range(nu):
            x = sweep(g, b, x, backward=False, colour_order=1)
            x = sweep(g, b, x, backward=True, colour_order=1)
    else:
        for _ in range(nu):
            x = sweep(g, b, x, backward=False, colour_order=1)
        r = b - O.addeval_node(g, 1.0, x) if node else O.addeval(g, -1.0, -1.0, x, b)
        bc = O.restrict_node(g, r) if node else O.restrict_edge(g, r)
        xc = cycle(gs, node, l - 1, bc, np.zeros_like(bc), nu, coarse, low)
        x = O.prolong_node(g, xc, x) if node else O.prolong_edge(g, xc, x)
        for _ in range(nu):
            x = sweep(g, b, x, backward=True, colour_order=1)
    low[l] = (b, x)
    return x


# 4 x 4 .. 12 x 12 coarse nodes (12: 288 edge unknowns, solved on the host; 3
# and 5: odd, no launch for the coarse end), rectangles, one to three sweeps,
# tops below, at and above the sizes that fit one launch or the LDS
@pytest.mark.parametrize("nx0,ny0,L,nu,coarse", [(4, 4, 1, 1, True), (4, 4, 3, 2, True), (4, 4, 5, 2, True),
                                                 (4, 8, 4, 3, True), (6, 6, 2, 2, False), (5, 3, 3, 2, True),
                                                 (12, 12, 2, 2, True), (10, 4, 3, 1, True)])
@pytest.mark.parametrize("node", [False, True])
def test_vcycle_every_level(M, nx0, ny0, L, nu, coarse, node):
    kx, ky, one = 0.4, -2.3, M.Cplx.of(1.0)
    nx, ny = nx0 << L, ny0 << L
    eta = 1.0 / np.random.default_rng(5).uniform(1.0, 9.0, size=(ny, nx))
    grids = [M.Grid(eta, kx, ky)]
    for _ in range(L):
        grids.insert(0, grids[0].coarse())
    for g in grids:
        g.set_bloch(kx, ky)
    kind = M.Node if node else M.Edge
    rng = np.random.default_rng(nx + nu)
    dim = nx * ny * (1 if node else 2)
    b, x = (rng.standard_normal(dim) + 1j * rng.standard_normal(dim) for _ in range(2))
    n0 = nx0 * ny0 * (1 if node else 2)
    A = None
    if coarse:
        A = M.lib.new_matrix(n0, n0)
        if node:
            M.lib.densematrix_node2d(True, grids[0].g, A)
        else:
            M.lib.densematrix_edge2d(one, one, grids[0].g, A)
        assert M.lib.potrf_matrix(A) == 0
    new = lambda: [kind(g, np.zeros(g.nx * g.ny * (1 if node else 2), complex)) for g in grids]
    B, X, D = new(), new(), new()
    B[L].set(b)
    X[L].set(x)
    (M.lib.vcycle_node2d if node else M.lib.vcycle_edge2d)(L, nu, A, arr(B), arr(X), arr(D))

    gs = [O.Grid2D(eta, kx=kx, ky=ky)]
    for _ in range(L):
        gs.insert(0, gs[0].coarse())
    low = {}
    cycle(gs, node, L, b, x, nu, coarse, low)
    # Every level's residual rounds at eps times its operator's row sum times
    # |x|: 8 eta / h^2 for the edges (the sum over levels of a quarter each and
    # both ways: below 40 / h^2), O(1) for the nodes.
    eps, h = 2.2e-16, min(gs[L].hx, gs[L].hy)
    tol = 500 * (L + 1) * eps if node else 40 * eps / (h * h)
    for l in range(L + 1):
        for got, ref in ((B[l].get(), low[l][0]), (X[l].get(), low[l][1])):
            err = np.abs(got - ref).max() / max(np.abs(ref).max(), np.abs(x).max())
            print("level %d err %.2e (tol %.2e)" % (l, err, tol))
            assert err <= tol, l
    if A:
        M.lib.del_matrix(A)
