"""Performance cases of the sparse path: products of CSR and block-CSR matrices with dense
blocks, CG and GMRES solves (one system, or many uneven ones in a batched engine) and the
assembly of CSR matrices from triples.

Every case runs through the public entry points with its operands resident on the GPU, as a
user's program holds them.  The matrices are the kinds the library is used with: grid
operators (2D / 3D graph Laplacians, plain or with log-normal edge coefficients, upwind
convection-diffusion) and matrices of uniformly scattered columns with Poisson row lengths.
"""
from __future__ import annotations

import ctypes
import math
import random

import torch

from tensors_amd import _capi as capi
from tensors_amd.batch import BatchCG, BatchGMRES
from tensors_amd.solvers import GMRES, ConjugateGradient, cg_solve_mixed, gmres_solve_mixed
from tensors_amd.sparse import KernelMatrixCSR, MatrixCSR

DEV = "cuda"
F64 = torch.float64
DTYPES = {"f64": torch.float64, "f32": torch.float32}

#: Relative residual that every solve reaches.
TOL = 1e-10
RESTART = 30
#: Rows of a block of `exact`'s per-system reductions.
CHUNK = 256


def listed():
    return [
        # The smallest call: one SpMV on a 256 x 256 grid operator, all of it in the caches.  What a
        # user's own iteration (a smoother, a time step) calls thousands of times.
        {"name": "spmv_grid2d_256_f64", "kind": "dot", "matrix": "grid2d", "rows": 65536, "cols": 65536, "mean": 5,
         "nrhs": 1, "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # The benchmark's random matrix, one and 64 right-hand sides: graph-like data, the columns of a
        # row anywhere in X.
        {"name": "spmv_random_1e6_f64", "kind": "dot", "matrix": "random", "rows": 1000000, "cols": 1000000,
         "mean": 32, "nrhs": 1, "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        {"name": "spmm_random_1e6_f64_k64", "kind": "dot", "matrix": "random", "rows": 1000000, "cols": 1000000,
         "mean": 32, "nrhs": 64, "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # Odd sizes: a rectangular matrix, 7 columns, FP32, an update of Y.
        {"name": "spmm_rect_f32_k7_update", "kind": "dot", "matrix": "random", "rows": 300007, "cols": 210001,
         "mean": 21, "nrhs": 7, "dtype": "f32", "alpha": -0.75, "beta": 0.5},
        # Block CSR as elasticity has it: 3 x 3 blocks on a 3D grid pattern.
        {"name": "bsr3_grid3d_96_f64_k4", "kind": "bsr", "side": 96, "block": 3, "nrhs": 4, "dtype": "f64"},
        # One right-hand side on a mid-size grid with varying coefficients, Jacobi: the launch-bound
        # solve of an implicit time step.
        {"name": "cg_weighted3d_45_jacobi", "kind": "cg", "side": 45, "nrhs": 1, "weighted": True, "mixed": False},
        # The largest solve: the benchmark's 128^3 Laplacian with 32 right-hand sides.
        {"name": "cg_laplacian3d_128_k32", "kind": "cg", "side": 128, "nrhs": 32, "weighted": False, "mixed": False},
        # Nonsymmetric solves, small (a request of the serving mix) in FP64 and large in mixed precision.
        {"name": "gmres_convdiff_100_f64", "kind": "gmres", "side": 100, "peclet": 3.0, "mixed": False},
        {"name": "gmres_convdiff_1000_mixed", "kind": "gmres", "side": 1000, "peclet": 10.0, "mixed": True},
        # Many uneven systems at once, as the serving loop has them: CG with 1-8 right-hand sides on
        # grids of 1e3-2e5 rows in mixed precision, and small GMRES systems.
        {"name": "batch_cg_64_mixed", "kind": "batch_cg", "systems": 64, "layout": 4004, "mode": 1},
        {"name": "batch_gmres_64", "kind": "batch_gmres", "systems": 64, "lo": 100, "hi": 100, "layout": 5005},
        # Assembly: the graph Laplacian of a 96^3 grid from its edges' contributions, four triples an
        # edge, duplicates summed.
        {"name": "triples_grid3d_96", "kind": "triples", "side": 96, "shuffled": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dot", "dot", "dot", "bsr", "cg", "cg", "gmres", "batch_cg", "batch_gmres", "triples"])
    if kind == "dot":
        matrix = rng.choice(["random", "random", "grid2d", "grid3d"])
        nrhs = rng.choice([1, _log_int(rng, 1, 64)])
        dtype = rng.choice(["f64", "f32"])
        alpha, beta = rng.choice([(1.0, 0.0), (-0.75, 0.5)])
        if matrix == "random":
            rows = _log_int(rng, 2000, 1000000)
            cols, mean = rng.choice([rows, _log_int(rng, 2000, 1000000)]), rng.randint(4, 32)
        else:
            dims = int(matrix[4])
            rows = cols = (_log_int(rng, 50, 1000) if dims == 2 else _log_int(rng, 13, 100)) ** dims
            mean = 2 * dims + 1
        return {"kind": kind, "matrix": matrix, "rows": rows, "cols": cols, "mean": mean, "nrhs": nrhs,
                "dtype": dtype, "alpha": alpha, "beta": beta}
    if kind == "bsr":
        block = rng.choice([2, 3, 4, 6, 8])
        return {"kind": kind, "side": _log_int(rng, 10, 240 // block), "block": block,
                "nrhs": rng.choice([1, 2, 3, 4, 6, 8]), "dtype": rng.choice(["f64", "f32"])}
    if kind == "cg":
        weighted = rng.random() < 0.5
        return {"kind": kind, "side": _log_int(rng, 12, 70 if weighted else 128),
                "nrhs": _log_int(rng, 1, 8 if weighted else 32), "weighted": weighted, "mixed": rng.random() < 0.5}
    if kind == "gmres":
        return {"kind": kind, "side": _log_int(rng, 40, 1000), "peclet": round(math.exp(rng.uniform(0, math.log(30))), 2),
                "mixed": rng.random() < 0.5}
    if kind == "batch_cg":
        return {"kind": kind, "systems": _log_int(rng, 4, 64), "layout": rng.randrange(1 << 20),
                "mode": rng.choice([0, 1, 2])}
    if kind == "batch_gmres":
        lo = _log_int(rng, 30, 100)
        return {"kind": kind, "systems": _log_int(rng, 4, 64), "lo": lo, "hi": rng.randint(lo, 110),
                "layout": rng.randrange(1 << 20)}
    return {"kind": kind, "side": _log_int(rng, 10, 96), "shuffled": rng.random() < 0.5}


# -- inputs (from the seed alone, on the GPU) ---------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(g, *shape, dtype=F64):
    return torch.rand(*shape, dtype=F64, device=DEV, generator=g).mul_(2).sub_(1).to(dtype)


class Rows:
    """A matrix of at most S entries a row: columns and values n x S (ascending columns where `mask`,
    value 0 elsewhere)."""

    def __init__(self, col, val, mask):
        self.col, self.val, self.mask = col, val, mask

    def csr(self):
        rp = torch.zeros(self.col.shape[0] + 1, dtype=torch.int64, device=DEV)
        torch.cumsum(self.mask.sum(1), 0, out=rp[1:])
        return rp.to(torch.int32), self.col[self.mask].to(torch.int32), self.val[self.mask]


def _grid(sides):
    """Node numbers, per axis (stride, coordinate, side), of a grid in lexicographic order."""
    n = math.prod(sides)
    v = torch.arange(n, device=DEV)
    axes, stride = [], n
    for s in sides:
        stride //= s
        axes.append((stride, (v // stride) % s, s))
    return v, axes


def _laplacian(sides, shift, g=None):
    """Graph Laplacian + shift; edge weights 1, or exp(N(0,1)) drawn from g."""
    v, axes = _grid(sides)
    n = v.numel()
    low, high, diag = [], [], torch.full((n,), shift, dtype=F64, device=DEV)
    for stride, x, side in axes:
        w = torch.ones(n, dtype=F64, device=DEV) if g is None else torch.randn(n, dtype=F64, device=DEV, generator=g).exp_()
        up = (x < side - 1).double().mul_(w)
        down = torch.zeros_like(up)
        down[stride:] = up[:n - stride] if stride < n else up[:0]
        diag += up + down
        low.append((v - stride, -down, x > 0))
        high.append((v + stride, -up, x < side - 1))
    cols = low + [(v, diag, torch.ones_like(v, dtype=torch.bool))] + high[::-1]
    mask = torch.stack([m for _, _, m in cols], 1)
    col = torch.where(mask, torch.stack([c for c, _, _ in cols], 1), v[:, None])
    return Rows(col, torch.stack([a for _, a, _ in cols], 1), mask)


def _convection_diffusion(side, peclet, theta=math.pi / 6):
    """5-point diffusion plus upwind convection of strength 2 P along (cos theta, sin theta)."""
    v, ((s0, i, _), (s1, j, _)) = _grid((side, side))
    bx, by = 2 * peclet * math.cos(theta), 2 * peclet * math.sin(theta)
    one = torch.ones(v.numel(), dtype=F64, device=DEV)
    mask = torch.stack([i > 0, j > 0, i >= 0, j < side - 1, i < side - 1], 1)
    col = torch.where(mask, torch.stack([v - s0, v - s1, v, v + s1, v + s0], 1), v[:, None])
    val = torch.stack([-(1 + by) * one, -(1 + bx) * one, (4 + bx + by) * one, -one, -one], 1)
    return Rows(col, torch.where(mask, val, torch.zeros_like(val)), mask)


def _random_csr(g, m, n, mean):
    """Poisson(mean) entries a row (at least one, at most 512) in distinct uniform columns, N(0,1) values."""
    length = torch.poisson(torch.full((m,), float(mean), device=DEV), generator=g).clamp_(1, 512).long()
    row = torch.repeat_interleave(torch.arange(m, device=DEV), length)
    key = row * n + torch.randint(0, n, (row.numel(),), device=DEV, generator=g)
    key = torch.unique_consecutive(torch.sort(key)[0])
    rp = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(key // n, minlength=m), 0, out=rp[1:])
    val = torch.randn(key.numel(), dtype=F64, device=DEV, generator=g)
    return rp.to(torch.int32), (key % n).to(torch.int32), val


def _dot_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    if c["matrix"] == "random":
        rp, ci, val = _random_csr(g, c["rows"], c["cols"], c["mean"])
    else:
        dims = int(c["matrix"][4])
        rp, ci, val = _laplacian((round(c["rows"] ** (1 / dims)),) * dims, 1.0, g).csr()
    shape = ((c["cols"],), (c["rows"],)) if c["nrhs"] == 1 else ((c["cols"], c["nrhs"]), (c["rows"], c["nrhs"]))
    return rp, ci, val.to(dt), _uniform(g, *shape[0], dtype=dt), _uniform(g, *shape[1], dtype=dt)


def _bsr_inputs(c, seed):
    g, dt, b, k = _gen(seed), DTYPES[c["dtype"]], c["block"], c["nrhs"]
    rp, ci, _ = _laplacian((c["side"],) * 3, 1.0).csr()
    n = c["side"] ** 3
    A = _uniform(g, ci.numel(), b, b, dtype=dt)
    return rp, ci, A, _uniform(g, n, b, k, dtype=dt)


def _systems(c, seed):
    """The systems (matrix, B) of a solver case; a single solve is one of one."""
    g = _gen(seed)
    if c["kind"] == "cg":
        M = _laplacian((c["side"],) * 3, 1e-3 if c["weighted"] else 1e-2, g if c["weighted"] else None)
        return [(M, _uniform(g, c["side"] ** 3, c["nrhs"]))]
    if c["kind"] == "gmres":
        return [(_convection_diffusion(c["side"], c["peclet"]), _uniform(g, c["side"] ** 2, 1))]
    got = []
    for sides, k, peclet in _layout(c):
        M = _convection_diffusion(sides[0], peclet) if c["kind"] == "batch_gmres" else _laplacian(sides, 1e-3, g)
        got.append((M, _uniform(g, math.prod(sides), k)))
    return got


def _layout(c):
    """(sides, right-hand sides, Peclet number) of a batch's systems: CG systems of 1e3-2e5 rows (2D or
    3D, 1-8 right-hand sides), GMRES systems of side lo..hi, Peclet 1-100."""
    r, got = random.Random(c["layout"]), []
    for _ in range(c["systems"]):
        if c["kind"] == "batch_cg":
            n, dims = math.exp(r.uniform(math.log(1e3), math.log(2e5))), r.choice([2, 3])
            got.append(((max(2, round(n ** (1 / dims))),) * dims, r.randint(1, 8), 0.0))
        else:
            got.append(((r.randint(c["lo"], c["hi"]),) * 2, 1, math.exp(r.uniform(0, math.log(100)))))
    return got


def _jacobi(M):
    n = M.col.shape[0]
    return 1.0 / M.val[M.col.eq(torch.arange(n, device=DEV)[:, None]) & M.mask]


def _triples(c, seed):
    """(i, j, value) of every edge's four contributions, in the edges' order or shuffled."""
    g, (v, axes) = _gen(seed), _grid((c["side"],) * 3)
    I, J, V = [], [], []
    for stride, x, side in axes:
        a = v[x < side - 1]
        w = torch.randn(a.numel(), dtype=F64, device=DEV, generator=g).exp_()
        I.append(torch.stack([a, a, a + stride, a + stride], 1).reshape(-1))
        J.append(torch.stack([a, a + stride, a, a + stride], 1).reshape(-1))
        V.append(torch.stack([w, -w, -w, w], 1).reshape(-1))
    I, J, V = (torch.cat(x) for x in (I, J, V))
    if c["shuffled"]:
        p = torch.randperm(I.numel(), device=DEV, generator=g)
        I, J, V = I[p], J[p], V[p]
    return I.to(torch.int32), J.to(torch.int32), V


# -- what a user's program holds, and one pass ---------------------------------------------


def prepare(c, seed):
    kind = c["kind"]
    if kind == "dot":
        rp, ci, val, X, Y = _dot_inputs(c, seed)
        return {"case": c, "A": MatrixCSR.from_device(rp, ci, val, c["rows"], c["cols"]), "X": X, "Y": Y}
    if kind == "bsr":
        rp, ci, A, X = _bsr_inputs(c, seed)
        n = c["side"] ** 3
        K = KernelMatrixCSR(rp.cpu().numpy(), ci.cpu().numpy(), n, n, c["block"], c["block"])
        return {"case": c, "K": K, "A": A, "X": X, "Y": torch.empty_like(X)}
    if kind == "triples":
        I, J, V = _triples(c, seed)
        n, m = I.numel(), c["side"] ** 3
        ws = capi.lib().tg_csr_from_triples_workspace_bytes(n, m, 0)
        return {"case": c, "I": I, "J": J, "V": V, "rp": torch.empty(m + 1, dtype=torch.int32, device=DEV),
                "ci": torch.empty(n, dtype=torch.int32, device=DEV), "val": torch.empty(n, dtype=F64, device=DEV),
                "ws": torch.empty(ws, dtype=torch.uint8, device=DEV)}
    systems = _systems(c, seed)
    if kind in ("cg", "gmres"):
        M, B = systems[0]
        n, k = B.shape
        s = {"case": c, "A": MatrixCSR.from_device(*M.csr(), n, n), "B": B, "X": torch.zeros_like(B),
             "P": _jacobi(M) if c.get("weighted") else None}
        if c["mixed"]:
            s["a32"] = s["A"].device_arrays(torch.float32)[2]
        else:
            s["solver"] = ConjugateGradient(n, 20000, k) if kind == "cg" else GMRES(n, RESTART, k)
        return s
    X = torch.zeros(sum(B.numel() for _, B in systems), dtype=F64, device=DEV)
    parts, at = [], 0
    for M, B in systems:
        parts.append((*M.csr(), B, X[at:at + B.numel()].view_as(B), _jacobi(M) if kind == "batch_cg" else None))
        at += B.numel()
    return {"case": c, "engine": BatchCG() if kind == "batch_cg" else BatchGMRES(), "systems": parts, "X": X}


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "dot":
        s["A"].Dot(c["alpha"], s["X"], c["beta"], s["Y"])
        return s["Y"]
    if kind == "bsr":
        s["K"].Dot(s["A"], 1.0, s["X"], 0.0, s["Y"], c["nrhs"])
        return s["Y"]
    if kind == "triples":
        nnz = ctypes.c_int64(0)
        m, ws = c["side"] ** 3, s["ws"]
        capi.call("tg_csr_from_triples", s["I"].numel(), s["I"].data_ptr(), s["J"].data_ptr(), s["V"].data_ptr(),
                  capi.F64, m, m, 1, 0, s["rp"].data_ptr(), capi.I32, s["ci"].data_ptr(), s["val"].data_ptr(),
                  s["ci"].numel(), ws.data_ptr(), ws.numel(), ctypes.byref(nnz),
                  torch.cuda.current_stream().cuda_stream)
        return s["rp"], s["ci"][:nnz.value], s["val"][:nnz.value]
    if kind == "cg":
        if c["mixed"]:
            ok = cg_solve_mixed(s["A"], s["B"], s["X"], tol=TOL, P=s["P"], a32=s["a32"])[0]
        else:
            ok = s["solver"](s["A"], s["P"], 1.0, s["B"], 0.0, s["X"], TOL)
        return s["X"], int(ok)
    if kind == "gmres":
        if c["mixed"]:
            ok = gmres_solve_mixed(s["A"], s["B"], s["X"], tol=TOL, restart=RESTART, max_restarts=400, a32=s["a32"])[0]
        else:
            ok = s["solver"](s["A"], None, 1.0, s["B"], 0.0, s["X"], TOL, 400)
        return s["X"], int(ok)
    e, ids = s["engine"], []
    for rp, ci, val, B, X, d in s["systems"]:
        if kind == "batch_cg":
            ids.append(e.add(rp, ci, val, B, X, TOL, 20000, diag=d, mixed=c["mode"] == 1, true_residual=c["mode"] == 2))
        else:
            ids.append(e.add(rp, ci, val, B, X, TOL, restart=RESTART, max_restarts=400))
    e.run(16) if kind == "batch_cg" else e.run()
    good = 0
    for i in ids:
        good += int(e.result(i)["succeeded"])
        e.release(i)
    return s["X"], good


# -- what a pass cannot do without ---------------------------------------------------------


def _krylov(n, entries, k, size, vectors):
    """Bytes of one iteration: the matrix, `vectors` passes over n x k values."""
    return entries * (size + 4) + 4 * (n + 1) + vectors * n * k * size


def work(c):
    kind = c["kind"]
    size = 4 if c.get("dtype") == "f32" else 8
    if kind == "dot":
        nnz, k = c["rows"] * c["mean"], c["nrhs"]
        y = c["rows"] * k * size * (2 if c["beta"] else 1)
        return {"bytes": nnz * (size + 4) + 4 * (c["rows"] + 1) + c["cols"] * k * size + y, "flops": 2 * nnz * k}
    if kind == "bsr":
        n, b, k = c["side"] ** 3, c["block"], c["nrhs"]
        nnz = 7 * n - 6 * c["side"] ** 2
        return {"bytes": nnz * (b * b * size + 4) + 4 * (n + 1) + 2 * n * b * k * size, "flops": 2 * nnz * b * b * k}
    if kind == "triples":
        n = c["side"] ** 3
        count = 12 * (n - c["side"] ** 2)
        return {"bytes": 16 * count + 12 * (7 * n - 6 * c["side"] ** 2) + 4 * n, "flops": count}
    # Solves: an iteration reads the matrix and the direction and writes the product, reads and writes
    # x, r and the direction (8 passes more in all, as CG has them), or reads half a restart length of
    # basis vectors (GMRES).  The iterations are about what the operators of these sizes take to 1e-10.
    total, flops = 0, 0
    mixed = c.get("mixed") or c.get("mode") == 1
    size = 4 if mixed else 8
    if kind == "cg":
        parts = [((c["side"],) * 3, c["nrhs"], 0.0)]
    elif kind == "gmres":
        parts = [((c["side"],) * 2, 1, c["peclet"])]
    else:
        parts = _layout(c)
    for sides, k, _ in parts:
        n, entries = math.prod(sides), (2 * len(sides) + 1) * math.prod(sides)
        if "gmres" in kind:
            iters, vectors = 3 * sides[0] + 100, 2 + RESTART // 2
        else:
            hard = kind == "batch_cg" or c["weighted"]
            iters, vectors = min(1200, (8 if hard else 3) * sides[0]), 10 + (2 / k if hard else 0)
        total += iters * _krylov(n, entries, k, size, vectors)
        flops += iters * (2 * entries * k + 2 * vectors * n * k)
    return {"bytes": total, "flops": flops}


def tolerance(c):
    kind = c["kind"]
    if kind in ("dot", "bsr"):
        # sums of 5-32 products; measured 7e-8 and 2.4e-16 off the sum in 64 bits
        return {"rel": 4e-7, "max": 4e-6} if c["dtype"] == "f32" else {"rel": 1e-15, "max": 1e-14}
    if kind == "triples":
        return {"rel": 1e-15, "max": 1e-15}
    # A solve stops where its residual crosses 1e-10: another rounding may stop it a step earlier or later.
    # Measured 2e-10 to 1.3e-9 off A^-1 B (the drawn grids' condition numbers reach a few times the listed).
    return {"rel": 2e-8, "max": 2e-7}


# -- the same in 64 bits ---------------------------------------------------------------------


def _exact_dot(c, seed):
    rp, ci, val, X, Y = _dot_inputs(c, seed)
    m, k = c["rows"], c["nrhs"]
    X, out = X.double().reshape(-1, k), (c["beta"] * Y.double()).reshape(m, k)
    row = torch.repeat_interleave(torch.arange(m, device=DEV), (rp[1:] - rp[:-1]).long())
    step = max(1, (1 << 28) // k)
    for a in range(0, ci.numel(), step):
        part = slice(a, a + step)
        out.index_add_(0, row[part], (c["alpha"] * val[part].double())[:, None] * X[ci[part].long()])
    return out.reshape(Y.shape)


def _exact_bsr(c, seed):
    rp, ci, A, X = _bsr_inputs(c, seed)
    n, b, k = c["side"] ** 3, c["block"], c["nrhs"]
    row = torch.repeat_interleave(torch.arange(n, device=DEV), (rp[1:] - rp[:-1]).long())
    out, X = torch.zeros(n, b, k, dtype=F64, device=DEV), X.double()
    step = max(1, (1 << 27) // (b * b * k))
    for a in range(0, ci.numel(), step):
        part = slice(a, a + step)
        out.index_add_(0, row[part], (A[part].double()[:, :, :, None] * X[ci[part].long()][:, None]).sum(2))
    return out


def _exact_triples(c, seed):
    I, J, V = _triples(c, seed)
    m = c["side"] ** 3
    key, where = torch.unique(I.long() * m + J, return_inverse=True)
    val = torch.zeros(key.numel(), dtype=F64, device=DEV).index_add_(0, where, V)
    rp = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(key // m, minlength=m), 0, out=rp[1:])
    return rp.to(torch.int32), (key % m).to(torch.int32), val


class Stacked:
    """All systems of a case as one block-diagonal matrix with padded rows and columns, and sums and
    factors per system and column."""

    def __init__(self, systems):
        self.k = max(B.shape[1] for _, B in systems)
        self.rows, self.owner, col, val, B, at = [], [], [], [], [], 0
        slots = max(M.col.shape[1] for M, _ in systems)
        for i, (M, b) in enumerate(systems):
            n = b.shape[0]
            pad = -n % CHUNK
            col.append(torch.nn.functional.pad(M.col, (0, slots - M.col.shape[1], 0, pad)) + at)
            val.append(torch.nn.functional.pad(M.val, (0, slots - M.val.shape[1], 0, pad)))
            B.append(torch.nn.functional.pad(b, (0, self.k - b.shape[1], 0, pad)))
            self.rows.append((at, n, b.shape[1]))
            self.owner += [i] * ((n + pad) // CHUNK)
            at += n + pad
        self.col, self.val, self.B = torch.cat(col).t().contiguous(), torch.cat(val).t().contiguous(), torch.cat(B)
        self.owner = torch.tensor(self.owner, device=DEV)
        self.count = len(systems)

    def mul(self, x):
        y = self.val[0][:, None] * x[self.col[0]]
        for c, a in zip(self.col[1:], self.val[1:]):
            y.addcmul_(a[:, None], x[c])
        return y

    def dot(self, x, y):
        parts = (x * y).view(-1, CHUNK, self.k).sum(1)
        return torch.zeros(self.count, self.k, dtype=F64, device=DEV).index_add_(0, self.owner, parts)

    def scaled(self, f, x):
        return (x.view(-1, CHUNK, self.k) * f[self.owner][:, None]).view_as(x)

    def take(self, x):
        return [x[a:a + n, :k] for a, n, k in self.rows]


def _ratio(a, b):
    return torch.where((a == 0) | (b == 0), torch.zeros_like(a), a / torch.where(b == 0, torch.ones_like(b), b))


def _solved(S, symmetric, goal=1e-13):
    """A^-1 B by CG (Jacobi) or BiCGSTAB, started again from the true residual until it is below goal."""
    x, bb = torch.zeros_like(S.B), S.dot(S.B, S.B)
    n = S.B.shape[0]
    d = (S.val * (S.col == torch.arange(n, device=DEV))).sum(0)
    d = torch.where(d == 0, torch.ones_like(d), 1.0 / d)[:, None]
    for _ in range(12):
        r = S.B - S.mul(x)
        if bool((S.dot(r, r) <= goal ** 2 * bb).all()):
            return x
        stop = (0.3 * goal) ** 2 * bb
        if symmetric:
            z = d * r
            p, rz = z.clone(), S.dot(r, z)
            for i in range(3000):
                u = S.mul(p)
                alpha = _ratio(rz, S.dot(p, u))
                x += S.scaled(alpha, p)
                r -= S.scaled(alpha, u)
                rr = S.dot(r, r)
                if i % 16 == 15 and bool((rr <= stop).all()):
                    break
                z = d * r
                new = torch.where(rr <= stop, torch.zeros_like(rr), S.dot(r, z))
                p = z + S.scaled(_ratio(new, rz), p)
                rz = new
        else:
            r0, p = r.clone(), r.clone()
            rho = S.dot(r0, r)
            for i in range(600):
                y = d * p
                v = S.mul(y)
                alpha = _ratio(rho, S.dot(r0, v))
                s = r - S.scaled(alpha, v)
                z = d * s
                t = S.mul(z)
                omega = _ratio(S.dot(t, s), S.dot(t, t))
                x += S.scaled(alpha, y) + S.scaled(omega, z)
                r = s - S.scaled(omega, t)
                rr = S.dot(r, r)
                if i % 16 == 15 and bool((rr <= stop).all()):
                    break
                new = torch.where(rr <= stop, torch.zeros_like(rr), S.dot(r0, r))
                beta = _ratio(new, rho) * _ratio(alpha, omega)
                p = r + S.scaled(beta, p - S.scaled(omega, v))
                rho = new
    return None


def exact(c, seed):
    kind = c["kind"]
    if kind == "dot":
        return _exact_dot(c, seed)
    if kind == "bsr":
        return _exact_bsr(c, seed)
    if kind == "triples":
        return _exact_triples(c, seed)
    S = Stacked(_systems(c, seed))
    x = _solved(S, "cg" in kind)
    if x is None:
        return None
    parts = S.take(x)
    return (parts[0], 1) if kind in ("cg", "gmres") else (torch.cat([p.reshape(-1) for p in parts]), len(parts))
