"""The V-cycle's coarse levels in one workgroup against the same levels as
launches per colour: both compute every row in the same order, so the V-cycle
from any level and whole solves must give the same bits.

Grids: levels of 1 to 8 rows; odd coarse levels (column array) under even ones
(row patterns); 38 colours on the coarsest level; colours of more rows than the
workgroup has threads; levels just inside and outside the row limit; whole
hierarchies in one workgroup, whose rhs the mixed V-cycle reads in f64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [((16, 16, 16), 4), ((24, 16, 40), 4), ((32, 32, 32), 4), ((104, 40, 56), 4), ((256, 16, 16), 4),
         ((64, 64, 32), 3), ((20, 16, 15), 1), ((17, 9, 5), 1), ((2, 2, 2), 1), ((4, 6, 2), 2)]


@pytest.mark.parametrize("dims,nlevels", GRIDS)
def test_same_bits_as_launches_per_colour(hip, dims, nlevels):
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    rng = np.random.default_rng(8)
    r = hip.DeviceArray.from_host(rng.uniform(-1, 1, G.m))
    G.make_rhs(1, 21)

    def results():
        out = []
        for lv in range(nlevels):
            y = hip.DeviceArray.from_host(np.full(G.levels[lv].m, np.nan))   # overwritten, never read
            G.mg(r, y, level=lv)
            out.append(y.host())
        z = hip.DeviceArray(G.m, np.float32)
        G.mg_mixed(r, z)
        out.append(z.host())
        for mode in (hip.CG_F64, hip.CG_MIXED):
            G.vec["x"].upload(np.zeros(G.m))
            out.append(G.cg(max_iter=6, mode=mode)["history"])
            out.append(G.vec["x"].host())
        # the inner levels' buffers, as the last FP64 V-cycle left them
        y = hip.DeviceArray(G.m)
        G.mg(r, y)
        for lv in range(nlevels - 1):
            out.append(G.prolongation(y, level=lv).host())
        return out

    G.set_coarse_rows(0)
    want = results()
    for rows in (-1, 8191, 600):
        G.set_coarse_rows(rows)
        for k, (a, b) in enumerate(zip(results(), want)):
            assert np.array_equal(a, b), (dims, rows, k)
    # the same with the column array in place of the row patterns
    G.set_coarse_rows(-1)
    G.set_row_patterns(False)
    for k, (a, b) in enumerate(zip(results(), want)):
        assert np.array_equal(a, b), (dims, "columns", k)
    G.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_batch_same_bits(hip, mode):
    """The problems of a batch leave the launches together: with these row limits
    at level 2 (-1), at the coarsest (1000), at none (100)."""
    dims = [(16, 16, 16), (32, 32, 24), (64, 48, 40), (56, 72, 48), (64, 64, 64)]

    def results(rows):
        B = hip.Batch(dims, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
        for k, P in enumerate(B.problems):
            P.make_rhs(1, 60 + k)
            P.set_coarse_rows(rows)
        out = []
        for use_graph in (True, False):
            for P in B.problems:
                P.vec["x"].upload(np.zeros(P.m))
            B.cg(max_iter=5, mode=mode, use_graph=use_graph)
            out += [B.history(k) for k in range(len(dims))] + [P.vec["x"].host() for P in B.problems]
        B.close()
        return out

    want = results(0)
    for rows in (-1, 1000, 100):
        for a, b in zip(results(rows), want):
            assert np.array_equal(a, b), rows
