"""Performance cases of the solver: what a program that uses it spends its time on.

A case is one call path through the Python entry points at one grid: whole CG
solves (FP64 and mixed precision), a batch of uneven problems, the V-cycle
preconditioner, the zero-guess smoother, the sparse product and the vector
reductions.  Grids are those of the repository's own workloads (32^3, 104^3,
320^3, the 64-problem batch of nx, ny, nz from {16, 24, ..., 96}) and ragged
ones between them.

Vectors are in multicolour row order, as the entry points take them: the rows
of colour 0 in natural order, then colour 1, ... .  On every grid here the
colours are the eight parity classes of (ix, iy, iz), so a vector in that
order is eight strided slices of the natural (nz, ny, nx) array, one after the
other; the helpers below use nothing else, and `exact` works the whole V-cycle
and CG out on natural arrays in float64 with torch alone.
"""
import math

import numpy as np
import torch

import rochpcg_amd as hpcg

LEVELS = 4
# (pz, py, px) parity of the rows of colours 0..7
CLASSES = ((1, 1, 1), (0, 1, 1), (1, 0, 0), (0, 1, 0), (1, 0, 1), (0, 0, 1), (1, 1, 0), (0, 0, 0))


def listed():
    return [
        # the smallest call a CG written over the operators makes: one inner
        # product of 32^3 rows, result on the host
        dict(name="dot_32", path="dot", nx=32, ny=32, nz=32),
        # the smallest whole solve: 50 FP64 iterations at 32^3, launch-bound
        dict(name="cg_f64_32", path="cg", mode="f64", nx=32, ny=32, nz=32, iters=50, refine=0),
        # an ordinary mixed-precision solve on a small cube
        dict(name="cg_mixed_64", path="cg", mode="mixed", nx=64, ny=64, nz=64, iters=50, refine=0),
        # the reference's smallest benchmark size; its coarsest level is odd (13^3)
        dict(name="cg_f64_104", path="cg", mode="f64", nx=104, ny=104, nz=104, iters=50, refine=0),
        # the plain FP64 configuration at full size, ten iterations of a solve
        dict(name="cg_f64_320", path="cg", mode="f64", nx=320, ny=320, nz=320, iters=10, refine=0),
        # the mixed configuration at full size, the f64 true residual every ten iterations
        dict(name="cg_mixed_320", path="cg", mode="mixed", nx=320, ny=320, nz=320, iters=20, refine=10),
        # 64 independent uneven problems solved together to 1e-9
        dict(name="batch_f64", path="batch", mode="f64", count=64, seed=7),
        dict(name="batch_mixed", path="batch", mode="mixed", count=64, seed=7),
        # the operators on their own, for programs that bring their own Krylov
        # loop: the product on a ragged grid, the preconditioner in both
        # precisions, one smoother step
        dict(name="spmv_ragged", path="spmv", nx=200, ny=136, nz=184),
        dict(name="mg_f64_ragged", path="mg", mode="f64", nx=176, ny=96, nz=240),
        dict(name="mg_mixed_192", path="mg", mode="mixed", nx=192, ny=192, nz=192),
        dict(name="symgs_256", path="symgs_zero", nx=256, ny=256, nz=256),
    ]


def draw(rng):
    """A case of the listed paths on another grid: every side a multiple of 8
    (as a 4-level hierarchy needs), even and odd multiples alike, rows spread
    over the logarithm from 24^3 to 320^3 (a batch goes down to 16)."""
    path = rng.choice(("dot", "cg", "cg", "cg", "batch", "spmv", "mg", "mg", "symgs_zero"))
    mode = rng.choice(("f64", "mixed"))
    if path == "batch":
        return dict(path=path, mode=mode, count=rng.randint(4, 64), seed=rng.randint(1, 10 ** 6))

    def grid(side):
        dims = [side * math.exp(rng.uniform(-0.35, 0.35)) for _ in range(3)]
        scale = side / (dims[0] * dims[1] * dims[2]) ** (1.0 / 3.0)
        return [max(24, int(d * scale / 8 + 0.5) * 8) for d in dims]

    dims = grid(math.exp(rng.uniform(math.log(24), math.log(320))))
    while dims[0] * dims[1] * dims[2] > 320 ** 3:
        dims[dims.index(max(dims))] -= 8
    case = dict(path=path, nx=dims[0], ny=dims[1], nz=dims[2])
    if path in ("cg", "mg"):
        case["mode"] = mode
    if path == "cg":
        most = 10 if mode == "f64" else 20
        small = dims[0] * dims[1] * dims[2] <= 2 ** 21
        case["iters"] = rng.randint(20, 50) if small else rng.randint(5, most)
        case["refine"] = rng.choice((0, 10)) if mode == "mixed" else 0
    return case


# ---------------------------------------------------------------------------
# multicolour order and the 27-point operator on natural arrays


def _shape(case):
    return case["nz"], case["ny"], case["nx"]


def _to_colour(v):
    return torch.cat([v[pz::2, py::2, px::2].reshape(-1) for pz, py, px in CLASSES])


def _pad(v):
    out = torch.zeros([n + 2 for n in v.shape], dtype=v.dtype, device=v.device)
    out[1:-1, 1:-1, 1:-1] = v
    return out


def _neighbours(pad, cls, shape):
    """Sum over the 26 neighbours of the rows of one parity class; `pad` is the
    field with a border of zeros."""
    (pz, py, px), (nz, ny, nx) = cls, shape
    hz, hy, hx = (nz - pz + 1) // 2, (ny - py + 1) // 2, (nx - px + 1) // 2
    out = torch.zeros((hz, hy, hx), dtype=pad.dtype, device=pad.device)
    for dz in (0, 1, 2):
        for dy in (0, 1, 2):
            for dx in (0, 1, 2):
                if (dz, dy, dx) != (1, 1, 1):
                    z, y, x = pz + dz, py + dy, px + dx
                    out += pad[z:z + 2 * hz - 1:2, y:y + 2 * hy - 1:2, x:x + 2 * hx - 1:2]
    return out


def _apply(v):
    """A v: 26 on the diagonal, -1 for every neighbour in the grid."""
    pad, out = _pad(v), torch.empty_like(v)
    for cls in CLASSES:
        pz, py, px = cls
        out[pz::2, py::2, px::2] = 26.0 * v[pz::2, py::2, px::2] - _neighbours(pad, cls, v.shape)
    return out


def _smooth(r, x):
    """One symmetric Gauss-Seidel step in colour order: forward over the
    colours, then back from the last but one."""
    pad = _pad(x)
    inner = pad[1:-1, 1:-1, 1:-1]
    for cls in CLASSES + CLASSES[-2::-1]:
        pz, py, px = cls
        inner[pz::2, py::2, px::2] = (r[pz::2, py::2, px::2] + _neighbours(pad, cls, r.shape)) / 26.0
    return inner.clone()


def _vcycle(r, levels):
    x = _smooth(r, torch.zeros_like(r))
    if levels == 1:
        return x
    nz, ny, nx = (n // 2 * 2 for n in r.shape)
    even = (slice(0, nz, 2), slice(0, ny, 2), slice(0, nx, 2))
    xc = _vcycle((r - _apply(x))[even].contiguous(), levels - 1)
    x[even] += xc
    return _smooth(r, x)


def _cg(b, iters):
    x, r = torch.zeros_like(b), b.clone()
    history = [float(r.square().sum().sqrt())]
    for k in range(iters):
        z = _vcycle(r, LEVELS)
        rtz = float((r * z).sum())
        p = z if k == 0 else z + (rtz / old) * p
        old = rtz
        q = _apply(p)
        alpha = rtz / float((p * q).sum())
        x += alpha * p
        r -= alpha * q
        history.append(float(r.square().sum().sqrt()))
    return x, history


# ---------------------------------------------------------------------------
# inputs


def _field(seed, shape, salt):
    """Uniform in [-1, 1], as the repository's own workloads draw x*."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * salt + seed)
    return torch.rand(shape, generator=g, dtype=torch.float64, device="cuda") * 2.0 - 1.0


def _batch_dims(case):
    rng = np.random.RandomState(case["seed"])
    return [tuple(int(n) for n in rng.choice(np.arange(16, 97, 8), 3)) for _ in range(case["count"])]


class _Buffer:
    """A library vector as torch sees it."""

    def __init__(self, a):
        self.__cuda_array_interface__ = dict(shape=(a.n,), typestr=a.dtype.str, data=(a.ptr, False), version=2)


def _view(a):
    return torch.as_tensor(_Buffer(a), device="cuda")


def _stores(case):
    return hpcg.STORE_MIXED if case.get("mode") == "mixed" else hpcg.STORE_F64


def prepare(case, seed):
    """The hierarchy a program builds once and its vectors.  Solves have the
    right-hand side b = A x* of a drawn x*; the operators get a drawn vector,
    like a residual or a search direction."""
    path = case["path"]
    s = dict(case=case)
    if path == "batch":
        dims = _batch_dims(case)
        batch = hpcg.Batch(dims, nlevels=LEVELS, stores=_stores(case))
        s["batch"] = batch
        s["x"] = [_view(p.vec["x"]) for p in batch.problems]
        for k, (nx, ny, nz) in enumerate(dims):
            b = _apply(_field(seed, (nz, ny, nx), 3 + k))
            _view(batch.problems[k].vec["b"]).copy_(_to_colour(b))
    else:
        shape = _shape(case)
        s["problem"] = hpcg.Problem(case["nx"], case["ny"], case["nz"], nlevels=LEVELS, stores=_stores(case))
        v = _field(seed, shape, 1)
        if path == "cg":
            s["b"] = _to_colour(_apply(v))
            s["x"] = torch.zeros_like(s["b"])
            s["problem"].set_residual_replacement(case["refine"])
        else:
            s["v"] = _to_colour(v)
            kind = torch.float32 if path == "mg" and case["mode"] == "mixed" else torch.float64
            s["y"] = torch.zeros(s["v"].numel(), dtype=kind, device="cuda")
            if path == "dot":
                s["w"] = _to_colour(_field(seed, shape, 2))
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "batch":
        for x in s["x"]:
            x.zero_()
        torch.cuda.current_stream().synchronize()   # the batch runs on a stream of its own
        res = s["batch"].cg(max_iter=500, tol=1e-9, mode=hpcg.CG_MIXED if case["mode"] == "mixed" else hpcg.CG_F64)
        return dict(x=torch.cat(s["x"]), niters=res["niters"], normr0=res["normr0"])
    p = s["problem"]
    if path == "cg":
        s["x"].zero_()
        torch.cuda.current_stream().synchronize()   # the solver runs on a stream of its own
        res = p.cg(b=s["b"].data_ptr(), x=s["x"].data_ptr(), max_iter=case["iters"], tol=0.0,
                   mode=hpcg.CG_MIXED if case["mode"] == "mixed" else hpcg.CG_F64)
        return dict(x=s["x"], history=res["history"], niters=res["niters"])
    v, y = s["v"].data_ptr(), s["y"].data_ptr()
    if path == "dot":
        return p.dot(v, s["w"].data_ptr())
    if path == "spmv":
        p.spmv(v, y)
    elif path == "symgs_zero":
        p.symgs_zero(v, y)
    elif case["mode"] == "mixed":
        p.mg_mixed(v, y)
    else:
        p.mg(v, y)
    return s["y"]


def exact(case, seed):
    """The same results from natural arrays in float64.  A solve to a tolerance
    has the drawn solution as its limit."""
    path = case["path"]
    if path == "batch":
        xs = [_to_colour(_field(seed, (nz, ny, nx), 3 + k)) for k, (nx, ny, nz) in enumerate(_batch_dims(case))]
        return dict(x=torch.cat(xs), niters=None, normr0=None)
    shape = _shape(case)
    v = _field(seed, shape, 1)
    if path == "cg":
        if case["iters"] * v.numel() > 10 * 320 ** 3:
            return None   # over 20 s
        x, history = _cg(_apply(v), case["iters"])
        return dict(x=_to_colour(x), history=np.array(history), niters=None)
    if path == "dot":
        return float((v * _field(seed, shape, 2)).sum())
    if path == "spmv":
        return _to_colour(_apply(v))
    if path == "symgs_zero":
        return _to_colour(_smooth(v, torch.zeros_like(v)))
    return _to_colour(_vcycle(v, LEVELS))


# ---------------------------------------------------------------------------
# the work of one pass


def _smoother_work(m, nnz, vb, xb):
    # both triangles of the matrix once, r read, x written, then read and
    # written again on the way back
    return nnz * vb + 4 * m * xb, 4 * nnz


def _vcycle_work(dims, levels, vb, xb):
    m, nnz = math.prod(dims), math.prod(3 * n - 2 for n in dims)
    b, f = _smoother_work(m, nnz, vb, xb)
    if levels == 1:
        return b, f
    coarse = [n // 2 for n in dims]
    cb, cf = _vcycle_work(coarse, levels - 1, vb, xb)
    # the residual is needed, and the correction added, at the injected rows only
    rows = math.prod(coarse)
    return (2 * b + m * xb + rows * (27 * vb + 5 * xb) + cb, 2 * f + 54 * rows + cf)


def _iteration_work(dims, mode):
    m, nnz = math.prod(dims), math.prod(3 * n - 2 for n in dims)
    vb, xb = (2, 4) if mode == "mixed" else (8, 8)
    b, f = _vcycle_work(dims, LEVELS, vb, xb)
    # A p with p'Ap, r'z, p = z + beta p, x += alpha p, r -= alpha Ap with ||r||
    return b + nnz * vb + m * (16 + 8 + xb + xb + 32 + 24), f + 2 * nnz + 12 * m


def work(case):
    """Bytes and flops of one pass.  The matrix counts by its stored values,
    nonzeros only; it and the vectors are read again by every operator that
    needs all of them anew (each half of a smoother step, the residual, the
    product), since they outgrow the caches at every size where bytes decide."""
    path = case["path"]
    if path == "batch":
        # the problems take about 15 to 50 iterations to 1e-9, each its own
        # count; 30 stands for them
        b = f = 0
        for dims in _batch_dims(case):
            ib, fl = _iteration_work(dims, case["mode"])
            b, f = b + 30 * ib, f + 30 * fl
        return dict(bytes=b, flops=f)
    dims = (case["nx"], case["ny"], case["nz"])
    m, nnz = math.prod(dims), math.prod(3 * n - 2 for n in dims)
    if path == "dot":
        return dict(bytes=16 * m, flops=2 * m)
    if path == "spmv":
        return dict(bytes=8 * nnz + 16 * m, flops=2 * nnz)
    if path == "symgs_zero":
        b, f = _smoother_work(m, nnz, 8, 8)
        return dict(bytes=b, flops=f)
    if path == "mg":
        b, f = _vcycle_work(dims, LEVELS, *((2, 4) if case["mode"] == "mixed" else (8, 8)))
        return dict(bytes=b, flops=f)
    b, f = _iteration_work(dims, case["mode"])
    return dict(bytes=case["iters"] * b, flops=case["iters"] * f)
