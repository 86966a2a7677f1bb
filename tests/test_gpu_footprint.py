"""What a solver holds on the device: with the direct lifting the node vectors of
the finest level only; the buffers of the node V-cycles come with their first
use (timing them), once, and solves give the same before and after."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,graphs", [(0, False), (1, False), (1, True)])
def test_node_buffers_come_with_their_use(prec, graphs):
    import maxwell_amd as M
    n0, L, P, m = 4, 5, 3, 8
    S = M.Solver(O.rod_eta(n0 << L), n0=n0, levels=L, precision=prec, block=m, max_problems=P, march_min=64, graphs=graphs)
    solve = lambda: S.solve([0.3, 1.0, 2.0], [0.2, 0.4, -1.0], neig=6, tol=1e-8, maxit=200, seed=4)
    a = solve()
    before = S.stats()["device_bytes"]
    for _ in range(2):
        for kind in (2, 3, 5, 15):
            assert S.time_kernel(kind, 1)[0] > 0
    after = S.stats()["device_bytes"]
    value = 16 if prec == 0 else 8
    nodes = [(n0 << l) ** 2 * P * m * value for l in range(L + 1)]
    assert after - before == 3 * sum(nodes) - 2 * nodes[-1]
    b = solve()
    assert np.array_equal(a["lam"], b["lam"]) and np.array_equal(a["iters"], b["iters"]) and a["converged"].all()
    assert S.stats()["device_bytes"] == after
    S.close()


def test_solvers_with_node_cycles_hold_them_from_the_start():
    import maxwell_amd as M
    S = M.Solver(O.rod_eta(32), n0=4, levels=3, block=4, max_problems=1, phase_kernels=True)
    r = S.solve([0.4], [0.2], neig=2, tol=1e-8, maxit=200)
    assert r["converged"].all()
    before = S.stats()["device_bytes"]
    assert S.time_kernel(2, 1)[0] > 0
    assert S.stats()["device_bytes"] == before
    S.close()
