"""Setup's scan of a level's rows: the row patterns are the distinct rows of each
colour (column offsets and descriptor), counted here from the arrays, at most 32 of
them or none; colours of at most 4096 rows are searched by one block, in one launch
for eight rounds, larger ones by a launch a round.  And the pinned slots that
problems share for their results."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(32, 32, 32), (34, 32, 32), (48, 40, 36), (64, 2, 2), (32, 2, 2), (17, 19, 21), (13, 13, 13), (12, 14, 9),
         (5, 4, 3), (2, 2, 2)]


@pytest.mark.parametrize("dims", GRIDS)
def test_patterns_are_the_distinct_rows(hip, dims):
    G = hip.Problem(*dims, nlevels=1, stores=hip.STORE_F64)
    A, (_, off, _) = G.level_arrays(0), G.color_table(0)
    col = A["ell_col"]
    rows = np.where(col < 0, 0, col - np.arange(G.m)[:, None])
    rows = np.concatenate([rows, A["desc"][:, None]], axis=1)
    distinct = [len(np.unique(rows[off[c]:off[c + 1]], axis=0)) for c in range(G.levels[0].ncolors)]
    assert G.get_routes(0)[0] == (max(distinct) if max(distinct) <= 32 else 0)
    c = G.check_problem(0)
    assert not any(c[f] for f in ("perm", "color", "ell", "value", "desc")), c
    G.close()


def test_results_of_many_problems(hip):
    """More problems than a page has slots, used by several threads and given up in
    another order: each call returns its own result."""
    rng = np.random.default_rng(23)
    v = rng.integers(-8, 9, 512).astype(np.float64)   # sums of integers: exact in any order
    d = hip.DeviceArray.from_host(v)
    live = [hip.Problem(8, nlevels=1) for _ in range(70)]
    wrong = []

    def use(some):
        for k in some:
            for n in (512, 1 + k, 300 + k):
                got = live[k].dot(d, d, n)
                if got != float(np.dot(v[:n], v[:n])):
                    wrong.append((k, n, got))
    for _ in range(3):
        threads = [threading.Thread(target=use, args=(range(t, 70, 4),)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
        for k in rng.permutation(70)[:40]:
            live[k].close()
            live[k] = hip.Problem(8, nlevels=1)
    for P in live:
        P.close()
