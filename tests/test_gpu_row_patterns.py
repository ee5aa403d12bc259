"""Row patterns against the column array: both give a kernel the same columns in
the same slots, so every operator must give the same bits from either.

Grids: even on every level; odd coarse levels (which keep the column array);
two-row coarsest levels; one of 38 colours; single odd levels whose last slice,
block and wave are partial."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [((32, 32, 32), 4), ((24, 16, 40), 4), ((16, 16, 16), 4), ((256, 16, 16), 4), ((136, 72, 8), 3),
         ((17, 9, 5), 1), ((2, 2, 2), 1), ((64, 2, 6), 1)]


def _operators(hip, G, r, x0):
    out = []
    for lv, L in enumerate(G.levels):
        dr = hip.DeviceArray.from_host(r[:L.m])
        dx = hip.DeviceArray.from_host(x0[:L.m])
        y = hip.DeviceArray.from_host(np.full(L.m, np.nan))   # overwritten, never read
        G.spmv(dx, y, level=lv)
        out.append(y.host())
        G.symgs_zero(dr, y, level=lv)
        out.append(y.host())
        G.mg(dr, y, level=lv)
        out.append(y.host())
        G.symgs(dr, dx, level=lv)
        out.append(dx.host())
        if lv + 1 < G.nlevels:
            out.append(G.restriction(dr, dx, level=lv).host())
    z = hip.DeviceArray(G.m, np.float32)
    G.mg_mixed(hip.DeviceArray.from_host(r), z)
    out.append(z.host())
    for mode in (hip.CG_F64, hip.CG_MIXED):
        G.vec["x"].upload(np.zeros(G.m))
        out.append(G.cg(max_iter=6, mode=mode)["history"])
        out.append(G.vec["x"].host())
    return out


@pytest.mark.parametrize("dims,nlevels", GRIDS)
@pytest.mark.parametrize("shape", [(256, 1), (64, 2)])
def test_same_bits_as_the_column_array(hip, dims, nlevels, shape):
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    for mixed in (False, True):
        G.set_shape(*shape, mixed=mixed)
    rng = np.random.default_rng(5)
    r, x0 = rng.uniform(-1, 1, G.m), rng.uniform(-1, 1, G.m)
    got = _operators(hip, G, r, x0)
    G.set_row_patterns(False)
    want = _operators(hip, G, r, x0)
    for k, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a, b), (dims, shape, k)
    for lv in range(nlevels):
        c = G.check_problem(lv)
        assert not any(c[f] for f in ("perm", "color", "ell", "value", "desc")), (lv, c)
    G.close()


def test_unused_slots_keep_special_values_out(hip):
    """A row reads nothing from a slot it does not use: an infinity or a NaN in
    x reaches exactly the rows that have it as a neighbour."""
    dims = (32, 24, 16)
    G = hip.Problem(*dims, nlevels=1)
    x = np.random.default_rng(6).uniform(-1, 1, G.m)
    x[[0, 77, G.m - 1]] = [np.inf, np.nan, -np.inf]
    dx, y = hip.DeviceArray.from_host(x), hip.DeviceArray(G.m)
    out = []
    for on in (True, False):
        G.set_row_patterns(on)
        G.spmv(dx, y)
        a = y.host()
        G.symgs_zero(dx, y)
        out.append((a, y.host()))
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
    G.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_batch_same_bits(hip, mode):
    """Batched launches whose problems all have patterns, and ones (odd coarse
    levels among them) that fall back to the column array."""
    dims = [(32, 16, 48), (24, 40, 16), (16, 16, 16), (96, 16, 16)]
    hist = []
    for on in (True, False):
        B = hip.Batch(dims, stores=hip.STORE_F64 | hip.STORE_MIXED)
        for k, P in enumerate(B.problems):
            P.make_rhs(1, 40 + k)
            P.set_row_patterns(on)
        B.cg(max_iter=6, mode=mode)
        hist.append([B.history(k) for k in range(len(dims))] + [P.vec["x"].host() for P in B.problems])
        B.close()
    for a, b in zip(*hist):
        assert np.array_equal(a, b)
