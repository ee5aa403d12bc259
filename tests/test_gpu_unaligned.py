"""Callers' vectors need no more than their elements' alignment, also where an operator
takes two rows a thread (the defaults above 2^21 rows, or any level on request):
results from and into vectors one element behind an aligned address have the bits of
aligned ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,block", [((136, 128, 128), None), ((48, 32, 40), 64)])
def test_vectors_aligned_as_their_elements(hip, dims, block):
    G = hip.Problem(*dims, nlevels=2, stores=hip.STORE_F64 | hip.STORE_MIXED)
    if block:
        for mixed in (False, True):
            G.set_shape(block, 2, mixed=mixed)
    assert G.get_shape(0, hip.OP_SPMV)[1] == 2
    m = G.m
    rng = np.random.default_rng(14)
    v, x0 = rng.uniform(-1, 1, m), rng.uniform(-1, 1, m)

    def results(shift):
        def put(a):
            return hip.DeviceArray.from_host(np.concatenate([np.zeros(shift, a.dtype), a]))

        def at(d):
            return d.ptr + shift * d.dtype.itemsize
        out = []
        r, y = put(v), put(np.zeros(m))
        G.spmv(at(r), at(y))
        out.append(y.host()[shift:])
        for op in (G.symgs_zero, G.mg):
            op(at(r), at(y))
            out.append(y.host()[shift:])
        y = put(x0)
        G.symgs(at(r), at(y))
        out.append(y.host()[shift:])
        z = put(np.zeros(m, np.float32))
        G.mg_mixed(at(r), at(z))
        out.append(z.host()[shift:])
        for mode in (hip.CG_F64, hip.CG_MIXED):
            y = put(np.zeros(m))
            G.set_residual_replacement(2)
            out.append(G.cg(b=at(r), x=at(y), max_iter=3, tol=0.0, mode=mode)["history"])
            out.append(y.host()[shift:])
        return out

    for k, (a, b) in enumerate(zip(results(1), results(0))):
        assert np.array_equal(a, b), (dims, k)
    G.close()
