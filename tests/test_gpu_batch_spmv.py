"""The batched SpMV of more than 2^21 rows (two rows a thread where every colour is
even) gives each row the bits of the problem's own SpMV, in the preamble and in the
fused p'Ap of an iteration; the odd grid keeps one row a thread."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
def test_rows_of_large_batches(hip, mode, odd):
    dims = [(104, 104, 96), (96, 96, 104), (16, 24, 16), (88, 56, 40)] + [(17, 19, 21)] * odd
    B = hip.Batch(dims, nlevels=1, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
    assert sum(P.m for P in B.problems) > 1 << 21
    rng = np.random.default_rng(12)
    for k, P in enumerate(B.problems):
        P.make_rhs(1, 40 + k)
        P.vec["x"].upload(rng.uniform(-1, 1, P.m))
    B.cg(max_iter=1, tol=0.0, mode=mode)
    for P in B.problems:
        y = hip.DeviceArray(P.m)
        P.spmv(P.vec["p"], y)
        P.synchronize()
        assert np.array_equal(P.vec["Ap"].host(), y.host())
    B.cg(max_iter=0, tol=0.0, mode=mode)   # r = b - A x of the last x
    for P in B.problems:
        y = hip.DeviceArray(P.m)
        P.spmv(P.vec["x"], y)
        P.synchronize()
        assert np.array_equal(P.vec["Ap"].host(), y.host())
    B.close()
