"""Every problem of a batch stops at the first iteration whose residual meets the
tolerance, whatever the host has queued behind it: solves of no iteration, of one,
cut off by max_iter, and of problems that stop at different ones; the scalars are
those of the history, and a second solve starts anew."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_stops_with_the_last_problem(hip, mode):
    dims = [(16, 16, 16), (32, 32, 24), (24, 40, 56), (64, 48, 40)]
    B = hip.Batch(dims, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
    for k, P in enumerate(B.problems):
        P.make_rhs(1, 90 + k)
    for tol, max_iter in ((2.0, 50), (0.3, 50), (1e-6, 50), (1e-6, 3), (1e-6, 2), (1e-6, 1), (1e-6, 0), (0.0, 4), (1e-6, 50)):
        for use_graph in (True, False):
            for P in B.problems:
                P.vec["x"].upload(np.zeros(P.m))
            r = B.cg(max_iter=max_iter, tol=tol, mode=mode, use_graph=use_graph)
            for k in range(len(dims)):
                n, h = int(r["niters"][k]), B.history(k)
                want = next(i for i in range(len(h)) if i >= max_iter or not h[i] / h[0] > tol)
                assert len(h) == n + 1 and n == want, (tol, max_iter, use_graph, k)
                assert r["normr"][k] == h[n] and r["normr0"][k] == h[0]
    B.close()
