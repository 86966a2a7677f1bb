"""Module-API cycles from two host threads, each with grids, vectors and coarse
matrices of its own.  The coarse factors and their inverses are kept for the
last matrix seen, so the threads' calls take turns replacing them (the larger
one's in a larger buffer); every call has to work with its own."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def arr(objs):
    return (C.c_void_p * len(objs))(*[o.h for o in objs])


class Problem:
    def __init__(self, M, n0, L, kx, ky):
        self.M, self.L = M, L
        n, one = n0 << L, M.Cplx.of(1.0)
        rng = np.random.default_rng(n0)
        grids = [M.Grid(1.0 / rng.uniform(1.0, 9.0, (n, n)), kx, ky)]
        for _ in range(L):
            grids.insert(0, grids[0].coarse())
        for g in grids:
            g.set_bloch(kx, ky)
        self.grids = grids
        self.edges = [[M.Edge(g, np.zeros(2 * g.nx * g.ny, complex)) for g in grids] for _ in range(3)]
        self.nodes = [[M.Node(g, np.zeros(g.nx * g.ny, complex)) for g in grids] for _ in range(3)]
        self.e0 = rng.standard_normal(2 * n * n) + 1j * rng.standard_normal(2 * n * n)
        self.e = M.Edge(grids[L])
        self.Ae, self.An = M.lib.new_matrix(2 * n0 * n0, 2 * n0 * n0), M.lib.new_matrix(n0 * n0, n0 * n0)
        M.lib.densematrix_edge2d(one, one, grids[0].g, self.Ae)
        M.lib.densematrix_node2d(True, grids[0].g, self.An)
        assert M.lib.potrf_matrix(self.Ae) == 0 and M.lib.potrf_matrix(self.An) == 0

    def run(self, calls):
        out = []
        b, x, d = (arr(v) for v in self.edges)
        nb, nx, nd = (arr(v) for v in self.nodes)
        for q in range(calls):
            self.e.set(self.e0)
            self.M.lib.pinvit_edge2d(self.L, 2, 1 + q % 2, 2, 7.5, self.e.h, self.Ae, b, x, d, self.An, nb, nx, nd)
            out.append(self.e.get())
        return out


def test_two_threads_with_different_coarse_matrices():
    import maxwell_amd as M
    problems = [Problem(M, 4, 3, 0.4, -1.1), Problem(M, 6, 2, -0.8, 2.0)]
    alone = [p.run(2) for p in problems]
    got = [None, None]

    def work(i):
        got[i] = problems[i].run(30)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        for q, e in enumerate(got[i]):
            # the same launches on the same values
            assert np.array_equal(e, alone[i][q % 2]), (i, q)
