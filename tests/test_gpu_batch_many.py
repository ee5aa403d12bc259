"""A batch whose SpMV takes more segments (one a problem and colour) than one launch
can name: 940 problems of seventy colours, 65 800 segments.  The problems at both
ends and beside the cut compute what the same problems do in a small batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS, COLOURS, COUNT = (64, 2, 2), 70, 940


def test_more_segments_than_one_launch(hip):
    cut = 65535 // COLOURS
    picked = [0, 1, cut - 1, cut, cut + 1, COUNT - 1]
    B = hip.Batch([DIMS] * COUNT, nlevels=1, stores=hip.STORE_F64 | hip.STORE_MIXED)
    S = hip.Batch([DIMS] * len(picked), nlevels=1, stores=hip.STORE_F64 | hip.STORE_MIXED)
    assert B.problems[0].levels[0].ncolors == COLOURS and COUNT * COLOURS > 65535
    for k, P in enumerate(B.problems):
        P.make_rhs(1, k)
    for k, P in zip(picked, S.problems):
        P.make_rhs(1, k)
    for mode in (hip.CG_F64, hip.CG_MIXED):
        for P in B.problems + S.problems:
            P.vec["x"].upload(np.zeros(P.m))
        r = B.cg(max_iter=3, tol=0.0, mode=mode)
        S.cg(max_iter=3, tol=0.0, mode=mode)
        assert np.all(r["niters"] == 3) and np.all(r["normr"] < r["normr0"])
        for j, k in enumerate(picked):
            assert np.array_equal(B.history(k), S.history(j)), (mode, k)
            assert np.array_equal(B.problems[k].vec["x"].host(), S.problems[j].vec["x"].host()), (mode, k)
    B.close()
    S.close()
