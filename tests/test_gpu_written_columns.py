"""Columns and descriptors that a caller writes through a level's pointers are
followed, by the operators, the V-cycle, a CG solve captured before and a batch
planned before, as by launches over the column array; the other levels and programs
that only read keep their routes."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _edit(hip, G, level, through_c=False):
    """In every third row, another row of the same colour in place of the last upper
    neighbour; returns the level's columns (rows, 27) as written."""
    L = G.levels[level]
    off = G.color_table(level)[1]
    cols = G.level_arrays(level)["ell_col"]
    colour = np.searchsorted(off, np.arange(L.m), side="right") - 1
    for r in range(0, L.m, 3):
        c = cols[r, 26]
        if c > r and colour[c] != colour[r]:
            k = colour[c]
            others = np.setdiff1d(np.arange(off[k], off[k + 1]), cols[r])
            if others.size:
                cols[r, 26] = others[r % others.size]
    sliced = np.full((hip.ell_padded_rows(L.m), 27), -1, np.int32)
    sliced[:L.m] = cols
    flat = np.ascontiguousarray(sliced.reshape(-1, 128, 27).transpose(0, 2, 1)).reshape(-1)
    if through_c:
        ptrs = (C.c_void_p * 13)()
        assert hip.lib.hpcgx_level_arrays(G.h, level, ptrs) == 0
        hip.DeviceArray(flat.size, np.int32, ptr=ptrs[0], owner=False).upload(flat)
    else:
        G.level_views(level)["ell_col"].upload(flat)
    return cols


def _results(hip, G):
    r = hip.DeviceArray.from_host(np.random.default_rng(9).uniform(-1, 1, G.m))
    out = []
    for lv in range(G.nlevels):
        y = hip.DeviceArray(G.levels[lv].m)
        G.spmv(r, y, level=lv)
        out.append(y.host())
        G.mg(r, y, level=lv)
        out.append(y.host())
        G.symgs(r, y, level=lv)
        out.append(y.host())
    z = hip.DeviceArray(G.m, np.float32)
    G.mg_mixed(r, z)
    out.append(z.host())
    for mode in (hip.CG_F64, hip.CG_MIXED):
        for use_graph in (True, False):
            G.vec["x"].upload(np.zeros(G.m))
            out.append(G.cg(max_iter=3, mode=mode, use_graph=use_graph)["history"])
    return out


@pytest.mark.parametrize("level,through_c", [(0, False), (1, True), (3, False)])
def test_written_columns_are_followed(hip, level, through_c):
    dims = (32, 24, 16)
    G, H = (hip.Problem(*dims, nlevels=4, stores=hip.STORE_F64 | hip.STORE_MIXED) for _ in range(2))
    for P in (G, H):
        P.make_rhs(1, 30)
    before = _results(hip, G)   # graphs are captured
    cols = _edit(hip, G, level, through_c)
    after = _results(hip, G)
    # the product against the written columns: two sums of 27 terms, the terms at most 52 in all
    m = G.levels[level].m
    x = np.random.default_rng(9).uniform(-1, 1, G.m)[:m]
    a = G.level_arrays(level)["ell_val"]
    want = (np.where(cols >= 0, a, 0.0) * x[np.maximum(cols, 0)]).sum(axis=1)
    assert np.abs(after[3 * level] - want).max() <= 2 * 27 * 52 * 2.0 ** -53
    assert not np.array_equal(after[3 * level], before[3 * level])
    # everything against launches over the column array
    _edit(hip, H, level)
    H.set_row_patterns(False)
    H.set_coarse_rows(0)
    for k, (p, q) in enumerate(zip(after, _results(hip, H))):
        assert np.array_equal(p, q, equal_nan=True), k
    G.close()
    H.close()


def test_readers_keep_the_patterns(hip):
    G = hip.Problem(32, stores=hip.STORE_F64)
    fast, ell = G.stream_bytes(), G.iteration_bytes()
    assert fast < ell
    V = G.level_views(0)
    V["perm"].host()
    V["ell_col"].host()
    G.level_arrays(0)
    assert G.stream_bytes() == fast
    assert V["ell_col"].ptr and G.stream_bytes() > fast     # an address to write at
    G.set_row_patterns(True, level=0)                       # as they were created
    assert G.stream_bytes() == fast
    G.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_written_columns_in_a_batch(hip, mode):
    dims = [(32, 16, 48), (24, 40, 16)]
    out = []
    for planned_first in (True, False):
        B = hip.Batch(dims, stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
        for k, P in enumerate(B.problems):
            P.make_rhs(1, 50 + k)
        if planned_first:
            B.cg(max_iter=2, mode=mode)
        for P in B.problems:
            P.vec["x"].upload(np.zeros(P.m))
            if not planned_first:
                P.set_row_patterns(False)
                P.set_coarse_rows(0)
        _edit(hip, B.problems[1], 0)
        B.cg(max_iter=3, mode=mode)
        out.append([B.history(k) for k in range(len(dims))] + [P.vec["x"].host() for P in B.problems])
        B.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)


def test_drop_in_layer(hip, tmp_path):
    """HPCGX_ReadColumnsInPlace: all columns of the finest level but the diagonal's
    cleared, A x is 26 x only if the product reads them where they lie."""
    exe = str(tmp_path / "written_columns")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include", "hpcg"),
                        os.path.join(ROOT, "tests", "cpp", "written_columns.cpp"), "-L" + os.path.join(ROOT, "rochpcg_amd"),
                        "-lrochpcg_amd", "-Wl,-rpath," + os.path.join(ROOT, "rochpcg_amd"), "-Wl,-rpath-link,/opt/rocm/lib", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["26", "26"]


def test_written_between_iterations(hip):
    """Pointers taken while iterations are queued: the graph is replaced behind them."""
    out = []
    for use_graph in (True, False):
        G = hip.Problem(32, 24, 16, nlevels=4, stores=hip.STORE_F64)
        G.make_rhs(1, 31)
        G.cg_begin(max_iter=8)
        G.cg_iterate(4, use_graph=use_graph)
        V = G.level_views(0)
        col = V["ell_col"].host()
        V["ell_col"].upload(col)   # the same columns, read in place from here
        G.cg_iterate(4, use_graph=use_graph)
        out.append(G.cg_end(hist_len=9)["history"])
        G.close()
    assert np.array_equal(*out) and len(out[0]) == 9
