"""The coarse workgroup reads the stored values that the launches read, and no others:
an infinite value in a slot that a sum does not use stays out of it, and where the
launches take the diagonal from the rows, so does the workgroup.  Both routes must give
the same bits, whatever the value arrays hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STORES = (("ell_val", "diag"), ("ell_f16", "diag_f16"))


def _diagonal_slots(G, level):
    """Where the diagonals of a level lie in its sliced ELL arrays."""
    r = np.arange(G.levels[level].m)
    return ((r // 128) * 27 + G.level_arrays(level)["diag_idx"]) * 128 + r % 128


def _vcycles(hip, G):
    r = hip.DeviceArray.from_host(np.random.default_rng(3).uniform(-1, 1, G.m))
    out = []
    for lv in range(G.nlevels):
        y = hip.DeviceArray(G.levels[lv].m)
        G.mg(r, y, level=lv)
        out.append(y.host())
    z = hip.DeviceArray(G.m, np.float32)
    G.mg_mixed(r, z)
    return out + [z.host()]


def _same_either_way(hip, G):
    G.set_coarse_rows(0)
    want = _vcycles(hip, G)
    for rows in (-1, 8191):
        G.set_coarse_rows(rows)
        for k, (a, b) in enumerate(zip(_vcycles(hip, G), want)):
            assert np.all(np.isfinite(b)) and np.array_equal(a, b), (rows, k)


@pytest.mark.parametrize("dims,nlevels", [((32, 32, 32), 4), ((48, 40, 32), 3), ((16, 16, 16), 2), ((20, 12, 8), 1)])
def test_infinite_unused_values_stay_out(hip, dims, nlevels):
    """Infinite diagonals in the last colour of the coarsest level: its rows become
    0, and the rows that do not use that slot stay finite."""
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    L = G.levels[nlevels - 1]
    last = int(G.color_table(nlevels - 1)[1][L.ncolors - 1])
    slots, V = _diagonal_slots(G, nlevels - 1), G.level_views(nlevels - 1)
    for ell, diag in STORES:
        a, d = V[ell].host(), V[diag].host()
        a[slots[last:]] = np.inf
        d[last:] = np.inf
        V[ell].upload(a)
        V[diag].upload(d)
    _same_either_way(hip, G)
    G.close()


@pytest.mark.parametrize("dims,nlevels", [((32, 32, 32), 4), ((64, 32, 48), 4), ((32, 2, 2), 2)])
def test_diagonals_of_the_rows(hip, dims, nlevels):
    """Diagonals changed in the rows alone, not in the array beside them; (32, 2, 2)
    injects rows of several colours, whose post-smoother reads whole rows."""
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    rng = np.random.default_rng(4)
    for lv in range(nlevels):
        slots, V = _diagonal_slots(G, lv), G.level_views(lv)
        for ell, _ in STORES:
            a = V[ell].host()
            a[slots] = rng.integers(20, 33, slots.size)
            V[ell].upload(a)
    _same_either_way(hip, G)
    G.close()


@pytest.mark.parametrize("dims,nlevels", [((32, 32, 32), 4), ((20, 12, 8), 1)])
def test_special_values_in_the_rhs(hip, dims, nlevels):
    """Infinities and NaN in r reach the rows that the launches let them reach; a
    one-level V-cycle may overwrite its rhs, also when it is run again."""
    G = hip.Problem(*dims, nlevels=nlevels, stores=hip.STORE_F64 | hip.STORE_MIXED)
    r = np.random.default_rng(5).uniform(-1, 1, G.m)
    special = r.copy()
    special[[3, G.m // 2, G.m - 2]] = [np.inf, np.nan, -np.inf]
    last = G.color_table(nlevels - 1)[1][G.levels[nlevels - 1].ncolors - 1]
    slots, V = _diagonal_slots(G, nlevels - 1), G.level_views(nlevels - 1)

    def results():
        out = []
        for rhs in (r, special):
            dr, y, z = hip.DeviceArray.from_host(rhs), hip.DeviceArray(G.m), hip.DeviceArray(G.m, np.float32)
            G.mg(dr, y)
            G.mg_mixed(dr, z)
            out += [y.host(), z.host()]
            if nlevels == 1:
                G.mg(dr, dr)
                out.append(dr.host())
        return out

    for infinite in (False, True):
        if infinite:
            a, d = V["ell_val"].host(), V["diag"].host()
            a[slots[last:]] = np.inf
            d[last:] = np.inf
            V["ell_val"].upload(a)
            V["diag"].upload(d)
        G.set_coarse_rows(0)
        want = results()
        G.set_coarse_rows(8191)
        for k, (a, b) in enumerate(zip(results(), want)):
            assert np.array_equal(a, b, equal_nan=True), (infinite, k)
    G.close()
