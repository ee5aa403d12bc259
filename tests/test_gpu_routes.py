"""The routes that must give the same bits -- row patterns against the column array,
the coarse workgroup against launches per colour -- with each shown to be the one that
ran: every level through the launches, batches whose problems differ in route, and the
largest levels that a workgroup's LDS and 16-bit offsets hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _vcycles(hip, G):
    r = hip.DeviceArray.from_host(np.random.default_rng(18).uniform(-1, 1, G.m))
    out = []
    for lv in range(G.nlevels):
        y = hip.DeviceArray(G.levels[lv].m)
        G.mg(r, y, level=lv)
        out.append(y.host())
        G.symgs(r, y, level=lv)
        out.append(y.host())
    z = hip.DeviceArray(G.m, np.float32)
    G.mg_mixed(r, z)
    return out + [z.host()]


def _same(a, b, *what):
    for k, (p, q) in enumerate(zip(a, b)):
        assert np.array_equal(p, q), (*what, k)


def test_defaults(hip):
    """32^3: all levels have patterns, those of at most 16^3 run in one workgroup;
    an odd level has none."""
    G = hip.Problem(32, stores=hip.STORE_F64 | hip.STORE_MIXED)
    for mixed in (False, True):
        routes = [G.get_routes(lv, mixed) for lv in range(4)]
        assert all(0 < n <= 32 for n, _ in routes)
        assert [w for _, w in routes] == [False, True, True, True]
    G.close()
    G = hip.Problem(104, nlevels=4, stores=hip.STORE_F64)
    assert G.get_routes(2)[0] > 0 and G.get_routes(3) == (0, True)   # 13^3
    assert not G.get_routes(3, mixed=True)[1]                        # no mixed store
    G.close()


@pytest.mark.parametrize("dims,nlevels", [((32, 32, 32), 4), ((24, 16, 40), 4), ((256, 16, 16), 4), ((136, 72, 8), 3)])
def test_patterns_on_every_level(hip, dims, nlevels):
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    G.set_coarse_rows(0)
    assert not any(G.get_routes(lv, mixed)[1] for lv in range(nlevels) for mixed in (False, True))
    used = [G.get_routes(lv)[0] > 0 for lv in range(nlevels)]
    assert used[0] and used[1]
    got = _vcycles(hip, G)
    G.set_row_patterns(False)
    assert not any(G.get_routes(lv)[0] for lv in range(nlevels))
    _same(got, _vcycles(hip, G), dims)
    G.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_batch_of_both_sources(hip, mode):
    """Every level as launches; on the coarsest one problem, of 13^3 rows, has no
    patterns, so that its launches read the column array for all."""
    dims = [(32, 16, 48), (104, 104, 104), (40, 40, 40)]
    out = []
    for on in (True, False):
        B = hip.Batch(dims, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
        for k, P in enumerate(B.problems):
            P.make_rhs(1, 40 + k)
            P.set_row_patterns(on)
            P.set_coarse_rows(0)
        pats = [[P.get_routes(lv, mixed=mode == 1)[0] > 0 for P in B.problems] for lv in range(4)]
        assert not on or (all(pats[0]) and any(pats[3]) and not all(pats[3]))
        B.cg(max_iter=5, mode=mode)
        out.append([B.history(k) for k in range(len(dims))] + [P.vec["x"].host() for P in B.problems])
        B.close()
    _same(*out)


@pytest.mark.parametrize("dims,nlevels,f64", [((14, 15, 39), 1, True), ((20, 20, 20), 3, True), ((40, 40, 40), 3, True),
                                              ((25, 15, 43), 1, False), ((21, 26, 30), 1, False), ((60, 52, 40), 2, False)])
def test_largest_levels_of_a_workgroup(hip, dims, nlevels, f64):
    """Up to 8191 rows in FP64 and 16383 mixed: 8190, 8000 (with two levels below it
    in LDS, and as a coarse level), 16125, 16380 and 15600."""
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    G.set_coarse_rows(16383)
    level = next(lv for lv in range(nlevels) if G.levels[lv].m <= (8191 if f64 else 16383))
    assert G.levels[level].m > (5000 if f64 else 8191)
    assert G.get_routes(level, mixed=not f64)[1] and not (f64 and G.m > 8191 and G.get_routes(0)[1])
    got = _vcycles(hip, G)
    G.set_coarse_rows(0)
    assert not G.get_routes(nlevels - 1, mixed=not f64)[1]
    _same(got, _vcycles(hip, G), dims)
    G.close()


def test_levels_past_the_workgroup(hip):
    """8192 rows in FP64, whose offsets need 17 bits, and 16384 mixed are launches
    whatever the limit."""
    G = hip.Problem(32, 16, 16, nlevels=1, stores=hip.STORE_F64 | hip.STORE_MIXED)
    G.set_coarse_rows(1 << 20)
    assert not G.get_routes(0)[1] and G.get_routes(0, mixed=True)[1]
    G.close()
    G = hip.Problem(32, 32, 16, nlevels=1, stores=hip.STORE_MIXED)
    G.set_coarse_rows(1 << 20)
    assert not G.get_routes(0, mixed=True)[1]
    G.close()
