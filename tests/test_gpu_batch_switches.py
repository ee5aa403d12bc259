"""A batch follows its problems' switches after it has been planned and solved: with
set_coarse_rows(0) every level's restriction is a launch of its own again, and the
results keep their bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_coarse_rows_of_a_planned_batch(hip, mode):
    dims = [(32, 32, 24), (16, 32, 48), (64, 48, 40)]
    B = hip.Batch(dims, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
    for k, P in enumerate(B.problems):
        P.make_rhs(1, 20 + k)

    def solve():
        out = []
        for use_graph in (True, False):
            for P in B.problems:
                P.vec["x"].upload(np.zeros(P.m))
            B.cg(max_iter=4, mode=mode, use_graph=use_graph)
            out += [P.vec["x"].host() for P in B.problems]
        return out, B.profile(iters=1, mode=mode)["restrict"][1]

    first, restricted = solve()
    B.problems[1].set_coarse_rows(0)   # the problems leave together: one keeps all
    second, all_levels = solve()
    assert all_levels > restricted
    for P in B.problems:
        P.set_coarse_rows(-1)
    third, again = solve()
    assert again == restricted
    for a, b, c in zip(first, second, third):
        assert np.array_equal(a, b) and np.array_equal(a, c)
    B.close()
