"""What this backend is timed on: the calls that its users' programs make, over the
sizes, value types and directions that they use.

A program holds its vectors in device memory (torch tensors here), builds a matrix
or a solver handle once and calls into the library many times. Each case is one
such call (or one step of a loop) through the Python binding of the C ABI:

  step          one sweep of a program's own solver loop written in primitives:
                y = A x, r = b - y, r.r to the host, x += w r
  mxv           one sparse product on a grid operator (27-point, constant or
                variable coefficients), FP64 or FP32
  unstructured  one product with a matrix without grid structure (ragged rows),
                plain or transposed
  cg            a conjugate gradient solve: to 1e-10, or a fixed number of iterations
  hpcg          a multigrid-preconditioned solve to 1e-10
  pagerank, bfs, khop   on R-MAT graphs
  batch         many small systems with several right-hand sides each, to 1e-8
  diff          forward and backward pass of a differentiable solve
"""
import ctypes
import math
import random  # noqa: F401  (draw's argument is a random.Random)

import numpy as np
import torch

import alp_amd as alp
from alp_amd import autograd

DEVICE = "cuda:0"
OFFSETS = [(dx, dy, dz) for dz in (0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)
           if dz > 0 or (dz == 0 and dy > 0) or (dz == 0 and dy == 0 and dx > 0)]
SHIFT = 1e-2


def listed():
    return [
        # the smallest call: a program's own loop on a small system, where latency,
        # launches and the scalar's way to the host count
        {"name": "step_16", "kind": "step", "nx": 16, "ny": 16, "nz": 16, "coefficients": "constant"},
        # the headline product: HPCG's system at 192^3, FP64, y += A x
        {"name": "mxv_192", "kind": "mxv", "nx": 192, "ny": 192, "nz": 192, "coefficients": "constant",
         "dtype": "f64", "accumulate": True},
        # a variable-coefficient operator on a grid with odd sides in FP32
        {"name": "mxv_101x75x61_f32", "kind": "mxv", "nx": 101, "ny": 75, "nz": 61, "coefficients": "variable",
         "dtype": "f32", "accumulate": False},
        # a matrix read from a file: ragged rows, no grid; the transposed direction
        {"name": "vxm_unstructured", "kind": "unstructured", "rows": 400009, "mean": 18.0, "spread": 0.8,
         "dtype": "f64", "transpose": True},
        # 50 iterations at 64^3 from a random start: the ordinary small solve
        {"name": "cg_64_50", "kind": "cg", "nx": 64, "ny": 64, "nz": 64, "coefficients": "constant",
         "precision": 0, "iterations": 50},
        # the headline solve: 192^3 to 1e-10, FP32 iterations with FP64 updates
        {"name": "cg_192_mixed", "kind": "cg", "nx": 192, "ny": 192, "nz": 192, "coefficients": "constant",
         "precision": 1, "iterations": 0},
        # HPCG's own solve at its benchmark size, mixed precision
        {"name": "hpcg_192_mixed", "kind": "hpcg", "nx": 192, "ny": 192, "nz": 192, "levels": 3, "precision": 1},
        # the same solver in FP64 on a small box
        {"name": "hpcg_88x56x40", "kind": "hpcg", "nx": 88, "ny": 56, "nz": 40, "levels": 2, "precision": 0},
        # web-graph ranking and traversal on a scale-22 R-MAT graph
        {"name": "pagerank_22", "kind": "pagerank", "scale": 22, "symmetric": True},
        {"name": "bfs_22", "kind": "bfs", "scale": 22, "symmetric": True},
        # 64 uneven systems with 8 right-hand sides each
        {"name": "batch_64x8", "kind": "batch", "systems": 64, "rhs": 8, "low": 16, "high": 96, "sides": 2024,
         "precision": 1},
        # a training step through the solver: forward, adjoint and the gradients
        {"name": "diff_128", "kind": "diff", "nx": 128, "ny": 128, "nz": 128, "precision": 0},
    ]


# ---- drawn cases ------------------------------------------------------------------


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _sides(rng, lo, hi, step=1):
    base = _log(rng, lo, hi)
    return [max(lo, min(hi, step * max(1, round(base * rng.uniform(0.7, 1.35) / step)))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["step", "mxv", "mxv", "unstructured", "cg", "cg", "hpcg", "hpcg", "pagerank", "bfs", "khop",
                       "batch", "diff"])
    if kind in ("step", "mxv", "cg"):
        nx, ny, nz = _sides(rng, 8, 192)
        c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "coefficients": rng.choice(["constant", "variable"])}
        if kind == "mxv":
            c.update(dtype=rng.choice(["f64", "f64", "f32"]), accumulate=rng.random() < 0.5)
        if kind == "cg":
            if c["coefficients"] == "variable":  # ten times the iterations of a constant operator
                nx, ny, nz = _sides(rng, 8, 112)
                c.update(nx=nx, ny=ny, nz=nz)
            # a fixed count stays below what convergence takes
            c.update(precision=rng.choice([0, 1, 3]),
                     iterations=rng.choice([0, 0, min(rng.randint(10, 100), max(nx, ny, nz))]))
        return c
    if kind == "unstructured":
        return {"kind": kind, "rows": int(_log(rng, 2000, 2000000)) | 1, "mean": round(_log(rng, 4, 60), 1),
                "spread": round(rng.uniform(0.0, 1.2), 2), "dtype": rng.choice(["f64", "f64", "f32"]),
                "transpose": rng.random() < 0.5}
    if kind == "hpcg":
        levels = rng.randint(1, 3)
        nx, ny, nz = _sides(rng, 16, 160, 2 ** levels)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "levels": levels, "precision": rng.choice([0, 1, 2])}
    if kind in ("pagerank", "bfs", "khop"):
        c = {"kind": kind, "scale": rng.randint(12, 22), "symmetric": rng.random() < 0.7,
             "degree": rng.randint(8, 16)}
        if kind == "khop":
            c["hops"] = rng.randint(1, 4)
        return c
    if kind == "batch":
        precision = rng.choice([0, 1])
        rhs = rng.choice([1, 2, 4, 8, 16])
        most = (256 if precision == 0 else 512) // rhs
        return {"kind": kind, "systems": int(_log(rng, 2, min(64, most) + 0.99)), "rhs": rhs, "low": 16,
                "high": rng.randint(32, 96), "sides": rng.randint(1, 10 ** 6), "precision": precision}
    nx, ny, nz = _sides(rng, 12, 112)
    return {"kind": "diff", "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice([0, 1])}


# ---- inputs ---------------------------------------------------------------------------


class Buffer:
    """A torch tensor where the binding takes a Vector (it reads these three)."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.n = tensor, tensor.data_ptr(), tensor.numel()
        self.dtype = np.dtype(str(tensor.dtype).replace("torch.", ""))


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _uniform(n, g, dtype=torch.float64):
    return torch.rand(n, generator=g, device=DEVICE, dtype=dtype)


def _normal(n, g, dtype=torch.float64):
    return torch.randn(n, generator=g, device=DEVICE, dtype=dtype)


def _theta(n, g):
    return torch.exp(_normal(13 * n, g))  # lognormal(0, 1) conductances


def _grid_matrix(case, g, flags=0):
    """The matrix of a grid case and its conductances (None: constant coefficients)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["coefficients"] == "constant":
        return alp.Matrix.stencil27(nx, ny, nz, flags=flags), None
    theta = _theta(nx * ny * nz, g)
    torch.cuda.synchronize()
    return alp.Matrix.conductance27(nx, ny, nz, theta.data_ptr(), SHIFT, flags), theta


def _unstructured(case, g):
    """Device CRS arrays of a square matrix: row lengths lognormal around the mean, half
    of a row's entries near the diagonal and half anywhere, columns ascending."""
    n = case["rows"]
    z = _normal(n, g)
    length = case["mean"] * torch.exp(case["spread"] * z - 0.5 * case["spread"] ** 2)
    length = length.round().clamp_(1, n).to(torch.int64)
    row = torch.repeat_interleave(torch.arange(n, device=DEVICE), length)
    m = row.numel()
    near = row + (_normal(m, g) * max(4.0, n / 200.0)).to(torch.int64)
    far = (_uniform(m, g) * n).to(torch.int64)
    col = torch.where(_uniform(m, g) < 0.5, near, far) % n
    key = torch.unique(row * n + col)  # sorted: rows in order, columns ascending
    row, col = torch.div(key, n, rounding_mode="floor"), key % n
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEVICE)
    off[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    val = _normal(key.numel(), g, torch.float32 if case["dtype"] == "f32" else torch.float64)
    return off, row, col, val


def _batch_sides(case):
    r = np.random.RandomState(case["sides"])
    return [r.randint(case["low"], case["high"] + 1, case["systems"]).astype(np.uint32) for _ in range(3)]


def _batch_rows(case):
    nx, ny, nz = (a.astype(np.int64) for a in _batch_sides(case))
    return int((nx * ny * nz).sum())


def prepare(case, seed):
    alp.init(0)
    g = _generator(seed)
    kind = case["kind"]
    s = {"case": dict(case)}
    if kind in ("step", "mxv", "cg", "hpcg", "diff"):
        n = case["nx"] * case["ny"] * case["nz"]
    if kind == "step":
        s["A"], s["theta"] = _grid_matrix(case, g)
        s["x"], s["b"] = Buffer(_uniform(n, g)), Buffer(_normal(n, g))
        s["y"], s["r"] = Buffer(torch.zeros_like(s["x"].tensor)), Buffer(torch.zeros_like(s["x"].tensor))
        s["weight"] = 1.0 / 64 if case["coefficients"] == "constant" else 1.0 / 1024
    elif kind == "mxv":
        f32 = case["dtype"] == "f32"
        s["A"], s["theta"] = _grid_matrix(case, g, alp.MAT_WITH_F32 if f32 else 0)
        t = torch.float32 if f32 else torch.float64
        s["x"], s["y"] = Buffer(_uniform(n, g, t)), Buffer(_normal(n, g, t))
        s["ring"] = alp.PLUS_TIMES_F32 if f32 else alp.PLUS_TIMES_F64
        s["descr"] = alp.DENSE | (0 if case["accumulate"] else alp.OVERWRITE)
    elif kind == "unstructured":
        f32 = case["dtype"] == "f32"
        off, row, col, val = _unstructured(case, g)
        idx = col.to(torch.int32)
        torch.cuda.synchronize()
        h = ctypes.c_void_p()
        alp.check(alp.lib().alp_hip_matrix_create_device(
            ctypes.byref(h), case["rows"], case["rows"], val.numel(), off.data_ptr(), idx.data_ptr(), val.data_ptr(),
            alp.VAL_F32 if f32 else alp.VAL_F64, alp.MAT_WITH_CCS if case["transpose"] else 0, None),
            "matrix_create_device")
        s["A"], s["triplets"] = alp.Matrix(h.value), (row, col, val)
        t = val.dtype
        s["x"], s["y"] = Buffer(_normal(case["rows"], g, t)), Buffer(torch.zeros(case["rows"], device=DEVICE, dtype=t))
        s["ring"] = alp.PLUS_TIMES_F32 if f32 else alp.PLUS_TIMES_F64
    elif kind == "cg":
        s["A"], s["theta"] = _grid_matrix(case, g, alp.MAT_WITH_F32 if case["precision"] else 0)
        s["solution"] = _uniform(n, g)
        s["b"] = torch.zeros_like(s["solution"])
        s["x"] = torch.zeros_like(s["solution"])
        s["x0"] = _uniform(n, g) if case["iterations"] else torch.zeros_like(s["solution"])
        torch.cuda.synchronize()
        alp.check(alp.mxv(Buffer(s["b"]), s["A"], Buffer(s["solution"])), "mxv")
    elif kind == "hpcg":
        s["H"] = alp.Hpcg(case["nx"], case["ny"], case["nz"], max_levels=case["levels"], colours=0,
                          f32=case["precision"] != 0)
        s["solution"] = _uniform(n, g)
        s["b"] = Buffer(_stencil_apply(s["solution"].view(case["nz"], case["ny"], case["nx"])).reshape(-1))
        s["x"] = Buffer(torch.zeros_like(s["solution"]))
    elif kind in ("pagerank", "bfs", "khop"):
        v = 1 << case["scale"]
        src, dst = alp.rmat_edges(case["scale"], case.get("degree", 16) * v, seed=int(seed) % (1 << 31) + 1)
        flags = alp.GRAPH_DROP_SELF_LOOPS | (alp.GRAPH_SYMMETRIZE if case["symmetric"] else 0)
        s["G"] = alp.graph_from_edges(v, src, dst, flags)
        src.free()
        dst.free()
        if kind == "pagerank":
            s["out"] = Buffer(torch.zeros(v, device=DEVICE, dtype=torch.float64))
        else:
            s["source"], _ = alp.max_degree_vertex(s["G"])
            s["out"] = Buffer(torch.zeros(v, device=DEVICE, dtype=torch.int32 if kind == "bfs" else torch.uint8))
    elif kind == "batch":
        nx, ny, nz = _batch_sides(case)
        k = case["systems"]
        coef = torch.exp(0.5 * _normal(3 * k, g)).cpu().numpy().reshape(3, k)  # lognormal(0, 0.5)
        s["coef"] = coef
        s["B"] = alp.Batch(nx, ny, nz, coef[0], coef[1], coef[2], case["rhs"])
        s["B"].autotune()
        s["b"] = Buffer(_normal(s["B"].nrows * case["rhs"], g))
        s["x"] = Buffer(torch.zeros_like(s["b"].tensor))
    else:
        s["theta"] = _theta(n, g).requires_grad_()
        s["b"] = _normal(n, g).requires_grad_()
        s["target"] = _normal(n, g)
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------------


def run(s):
    c = s["case"]
    kind = c["kind"]
    L = alp.lib()
    if kind == "step":
        A, x, y, b, r = s["A"], s["x"], s["y"], s["b"], s["r"]
        alp.check(alp.mxv(y, A, x, descr=alp.DENSE | alp.OVERWRITE), "mxv")
        alp.check(L.alp_hip_ewise_f64(x.n, 1, b.ptr, y.ptr, r.ptr), "ewise")
        norm2 = alp.dot(r, r)
        alp.check(L.alp_hip_axpy_f64(x.n, s["weight"], r.ptr, x.ptr), "axpy")
        return [x.tensor, norm2]
    if kind == "mxv":
        alp.check(alp.mxv(s["y"], s["A"], s["x"], s["ring"], s["descr"]), "mxv")
        return s["y"].tensor
    if kind == "unstructured":
        descr = alp.DENSE | alp.OVERWRITE
        if c["transpose"]:
            alp.check(alp.vxm(s["y"], s["x"], s["A"], s["ring"], descr), "vxm")
        else:
            alp.check(alp.mxv(s["y"], s["A"], s["x"], s["ring"], descr), "mxv")
        return s["y"].tensor
    if kind == "cg":
        x = s["x"]
        alp.check(L.alp_hip_memcpy_d2d(x.data_ptr(), s["x0"].data_ptr(), 8 * x.numel()), "copy of the start")
        if c["iterations"]:
            alp.cg(s["A"], s["b"].data_ptr(), x.data_ptr(), c["iterations"], 1e-300, c["precision"])
        else:
            alp.check(alp.cg(s["A"], s["b"].data_ptr(), x.data_ptr(), 100000, 1e-10, c["precision"])[0], "cg")
        return x
    if kind == "hpcg":
        x = s["x"]
        alp.check(L.alp_hip_set_f64(x.n, x.ptr, 0.0), "set")
        s["H"].solve(s["b"], x, 2000, 1e-10, c["precision"])
        return x.tensor
    if kind == "pagerank":
        it, q = ctypes.c_size_t(), ctypes.c_double()
        alp.check(L.alp_hip_pagerank(s["G"].h, s["out"].ptr, 0.85, 1e-9, 1000, ctypes.byref(it), ctypes.byref(q)),
                  "pagerank")
        return s["out"].tensor
    if kind == "bfs":
        _, levels, reached = alp.bfs(s["G"], s["source"], out=s["out"])
        return [s["out"].tensor, levels, reached]
    if kind == "khop":
        alp.khop(s["G"], s["source"], c["hops"], out=s["out"])
        return s["out"].tensor
    if kind == "batch":
        alp.check(s["B"].solve(s["b"], s["x"], 1e-8, 20000, c["precision"])[0], "batch_solve")
        return s["x"].tensor
    x = autograd.solve(s["theta"], s["b"], (c["nx"], c["ny"], c["nz"]), 1e-10, c["precision"], SHIFT)
    loss = ((x - s["target"]) ** 2).sum()
    dtheta, db = torch.autograd.grad(loss, (s["theta"], s["b"]))
    return [x.detach(), dtheta, db]


# ---- what a pass cannot do without ------------------------------------------------------


def _iterations(case):
    """About how many iterations a solve takes (measured at a few sizes)."""
    if case.get("iterations"):
        return case["iterations"]
    side = max(case["nx"], case["ny"], case["nz"])
    if case["kind"] == "hpcg":
        return 12 + 0.68 * side
    if case["kind"] == "diff" or case["coefficients"] == "variable":
        return 100 + 9.0 * side
    return 8 + 1.6 * side


def work(case):
    """Each input read once and each output written once. A constant-coefficient
    operator has no value stream (27 numbers); a variable one has a value per entry. A
    solve counts, for each iteration, the operator and the vectors that its recurrences
    read and write (x, r, p, A p: six reads and writes of a vector beside the product)."""
    kind = case["kind"]
    if kind in ("step", "mxv", "cg", "hpcg", "diff"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = nx * ny * nz
        nnz = (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    if kind == "step":
        return {"bytes": 8 * 9 * n + (8 * nnz if case["coefficients"] == "variable" else 0), "flops": 2 * nnz + 5 * n}
    if kind == "mxv":
        es = 4 if case["dtype"] == "f32" else 8
        return {"bytes": es * ((3 if case["accumulate"] else 2) * n +
                               (nnz if case["coefficients"] == "variable" else 0)), "flops": 2 * nnz}
    if kind == "unstructured":
        es = 4 if case["dtype"] == "f32" else 8
        m = case["rows"] * case["mean"]
        return {"bytes": (es + 4) * m + (2 * es + 4) * case["rows"], "flops": 2 * m}
    if kind in ("cg", "diff"):
        es = 8 if case["precision"] == 0 else 4
        it = _iterations(case) * (2 if kind == "diff" else 1)
        values = es * nnz if kind == "diff" or case["coefficients"] == "variable" else 0
        vectors = 8 * es * n + (8 * n if case["precision"] == 1 else 0)
        return {"bytes": it * (values + vectors), "flops": it * (2 * nnz + 10 * n)}
    if kind == "hpcg":
        # per iteration on the finest level: two symmetric sweeps (four passes over
        # z and r), the residual, the product and the CG vectors; 8/7 for the coarse levels
        es = 8 if case["precision"] == 0 else 4
        it = _iterations(case)
        return {"bytes": it * es * n * (4 * 3 + 3 + 8) * 8 / 7, "flops": it * (2 * nnz * 6 + 10 * n) * 8 / 7}
    if kind in ("pagerank", "bfs", "khop"):
        v = 1 << case["scale"]
        m = (1.9 if case["symmetric"] else 0.95) * case.get("degree", 16) * v
        if kind == "pagerank":
            return {"bytes": 45 * (4 * m + 8 * 5 * v), "flops": 45 * (m + 6 * v)}
        if kind == "bfs":
            return {"bytes": 0.1 * 4 * m + 4 * 4 * v, "flops": 0}
        return {"bytes": 0.1 * 4 * m + 5 * v, "flops": 0}
    rows = _batch_rows(case)
    es = 8 if case["precision"] == 0 else 4
    # the largest system sets the count; on average half of the rows are still active
    it = 0.5 * 4.3 * max(int(a.max()) for a in _batch_sides(case))
    return {"bytes": it * rows * case["rhs"] * es * 8, "flops": it * rows * case["rhs"] * 24}


def tolerance(case):
    """About four times what the present code differs by from exact(), or, for solves
    that stop at a residual, what two runs that stop an iteration apart differ by."""
    kind = case["kind"]
    if kind in ("bfs", "khop"):
        return "exact"
    if kind == "step":
        return {"rel": 1e-14, "max": 1e-12}
    if kind in ("mxv", "unstructured"):
        return {"rel": 6e-7, "max": 3e-5} if case["dtype"] == "f32" else {"rel": 2e-15, "max": 1e-13}
    if kind == "cg" and case["iterations"]:  # FP32 directions and residuals in the mixed modes
        return {"rel": 1e-12, "max": 1e-10} if case["precision"] == 0 else {"rel": 1e-5, "max": 1e-3}
    if kind in ("cg", "hpcg", "diff"):
        return {"rel": 1e-7, "max": 1e-5}
    if kind == "pagerank":
        return {"rel": 1e-9, "max": 1e-6}
    return {"rel": 2e-6, "max": 2e-4}


# ---- the same in 64 bits -----------------------------------------------------------------


def _box(t, axis):
    """Sum over a point and its two neighbours along an axis (zero outside)."""
    out = t.clone()
    m = t.shape[axis]
    out.narrow(axis, 1, m - 1).add_(t.narrow(axis, 0, m - 1))
    out.narrow(axis, 0, m - 1).add_(t.narrow(axis, 1, m - 1))
    return out


def _stencil_apply(u):
    return 27.0 * u - _box(_box(_box(u, 2), 1), 0)


def _pair(u, d):
    """The two ends of every edge along offset d = (dx, dy, dz)."""
    lo = hi = u
    for axis, step in ((2, d[0]), (1, d[1]), (0, d[2])):
        m = u.shape[axis] - abs(step)
        lo = lo.narrow(axis, max(0, -step), m)
        hi = hi.narrow(axis, max(0, step), m)
    return lo, hi


def _conductance_apply(theta, shape):
    parts = theta.view(*shape, 13)
    weights = [_pair(parts[..., k], d)[0].contiguous() for k, d in enumerate(OFFSETS)]

    def apply(u):
        out = SHIFT * u
        for w, d in zip(weights, OFFSETS):
            a, b = _pair(u, d)
            flow = w * (a - b)
            p, q = _pair(out, d)
            p += flow
            q -= flow
        return out

    return apply


def _operator(case, theta):
    shape = (case["nz"], case["ny"], case["nx"])
    if theta is None:
        return _stencil_apply, shape
    return _conductance_apply(theta.detach(), shape), shape


def _plain_cg(apply, b, x, iterations, tol):
    r = b - apply(x)
    p, rr = r.clone(), (r * r).sum()
    stop = float((b * b).sum()) * tol * tol
    for i in range(iterations):
        ap = apply(p)
        alpha = rr / (p * ap).sum()
        x = x + alpha * p
        r = r - alpha * ap
        new = (r * r).sum()
        if i % 16 == 15 and float(new) < stop:
            break
        p = r + (new / rr) * p
        rr = new
    return x


def _sines(n):
    k = torch.arange(1, n + 1, device=DEVICE, dtype=torch.float64)
    return math.sqrt(2.0 / (n + 1)) * torch.sin(math.pi / (n + 1) * k[:, None] * k[None, :]), \
        2.0 - 2.0 * torch.cos(math.pi / (n + 1) * k)


def _laplace_solve(shape, coef, b):
    """An anisotropic Dirichlet Laplacian solved in its sine basis; b: (nz, ny, nx, rhs)."""
    (sz, lz), (sy, ly), (sx, lx) = (_sines(m) for m in shape)

    def transform(t):
        nz, ny, nx, k = t.shape
        t = (sz @ t.reshape(nz, -1)).reshape(nz, ny, nx, k)
        t = (sy @ t.permute(1, 0, 2, 3).reshape(ny, -1)).reshape(ny, nz, nx, k).permute(1, 0, 2, 3)
        return (sx @ t.permute(2, 0, 1, 3).reshape(nx, -1)).reshape(nx, nz, ny, k).permute(1, 2, 0, 3)

    cx, cy, cz = coef
    lam = cz * lz[:, None, None] + cy * ly[None, :, None] + cx * lx[None, None, :]
    return transform(transform(b) / lam[..., None]).contiguous()


def _pagerank(G):
    off, idx, _ = G.download(0, with_values=False)
    off = torch.from_numpy(off.astype(np.int64)).to(DEVICE)
    col = torch.from_numpy(idx.view(np.int32)).to(DEVICE).to(torch.int64)
    n = off.numel() - 1
    deg = (off[1:] - off[:-1])
    row = torch.repeat_interleave(torch.arange(n, device=DEVICE), deg)
    scale = torch.where(deg > 0, 0.85 / deg.clamp(min=1).double(), torch.zeros(n, device=DEVICE, dtype=torch.float64))
    pr = torch.full((n,), 1.0 / n, device=DEVICE, dtype=torch.float64)
    for _ in range(1000):
        lost = pr[deg == 0].sum()
        new = torch.zeros_like(pr).index_add_(0, col, (pr * scale)[row]) + (0.85 * lost + 0.15) / n
        change = float((new - pr).abs().sum())
        pr = new
        if change <= 1e-9:
            break
    return pr


def exact(case, seed):
    kind = case["kind"]
    if kind in ("bfs", "khop"):
        return None
    s = prepare(case, seed)
    if kind == "step":
        apply, shape = _operator(case, s["theta"])
        x, b = s["x"].tensor.view(shape), s["b"].tensor.view(shape)
        r = b - apply(x)
        return [(x + s["weight"] * r).reshape(-1), float((r * r).sum())]
    if kind == "mxv":
        apply, shape = _operator(case, s["theta"])
        y = apply(s["x"].tensor.double().view(shape)).reshape(-1)
        return y + s["y"].tensor.double() if case["accumulate"] else y
    if kind == "unstructured":
        row, col, val = s["triplets"]
        if case["transpose"]:
            row, col = col, row
        y = torch.zeros(case["rows"], device=DEVICE, dtype=torch.float64)
        return y.index_add_(0, row, val.double() * s["x"].tensor.double()[col])
    if kind == "cg":
        if not case["iterations"]:
            return s["solution"]
        apply, shape = _operator(case, s["theta"])
        return _plain_cg(apply, s["b"].view(shape), s["x0"].view(shape), case["iterations"], 0.0).reshape(-1)
    if kind == "hpcg":
        return s["solution"]
    if kind == "pagerank":
        return _pagerank(s["G"])
    if kind == "batch":
        nx, ny, nz = _batch_sides(case)
        rows = [int(a) * int(b) * int(c) for a, b, c in zip(nx, ny, nz)]
        parts = torch.split(s["b"].tensor.view(-1, case["rhs"]), rows)
        out = [_laplace_solve((int(nz[k]), int(ny[k]), int(nx[k])), s["coef"][:, k],
                              p.view(int(nz[k]), int(ny[k]), int(nx[k]), case["rhs"])).reshape(-1)
               for k, p in enumerate(parts)]
        return torch.cat(out)
    apply, shape = _operator({**case, "coefficients": "variable"}, s["theta"])
    zero = torch.zeros(shape, device=DEVICE, dtype=torch.float64)
    x = _plain_cg(apply, s["b"].detach().view(shape), zero, 20000, 1e-13)
    lam = _plain_cg(apply, 2.0 * (x - s["target"].view(shape)), zero, 20000, 1e-13)
    grad = torch.zeros(*shape, 13, device=DEVICE, dtype=torch.float64)
    for k, d in enumerate(OFFSETS):
        (xa, xb), (la, lb) = _pair(x, d), _pair(lam, d)
        _pair(grad[..., k], d)[0].copy_(-(la - lb) * (xa - xb))
    return [x.reshape(-1), grad.reshape(-1), lam.reshape(-1)]
