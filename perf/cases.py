"""Timed cases of the framework's main paths.

What a program built on ``numml_amd.sparse`` spends its time in: matrix-vector and
matrix-matrix products with gradients (solvers and graph layers), sparse products (two-hop
graphs, coarse-grid operators), sums of matrices, triangular solves and direct solves.
``listed()`` names twelve of them, ``draw(rng)`` makes more out of the same ranges.

Matrices are the ones such programs assemble: five-point and seven-point stencils on grids of
any side lengths, and graphs with power-law degrees whose columns are uniformly random.
Everything is made on the GPU from the seed.
"""
import math

import torch

from numml_amd import sparse as sp
from numml_amd.sparse import linalg

DTYPES = {"f32": torch.float32, "f64": torch.float64}


# ---- the cases ---------------------------------------------------------------------

def listed():
    return [
        # one operator application and its gradients on a small grid: launches and host work
        {"name": "spmv_grid2d_small", "family": "spmv", "kind": "grid2d", "nx": 256, "ny": 256,
         "dtype": "f64", "grad": True},
        # the same on a grid of 4 M unknowns: a learned stencil, gradients of its values and of x
        {"name": "spmv_grid2d_large", "family": "spmv", "kind": "grid2d", "nx": 2048, "ny": 2048,
         "dtype": "f32", "grad": True},
        # the matrix-vector product inside an iterative solver, no gradients
        {"name": "spmv_grid3d_apply", "family": "spmv", "kind": "grid3d", "nx": 127, "ny": 113, "nz": 101,
         "dtype": "f64", "grad": False},
        # a graph layer's neighbourhood sum on a large graph, training
        {"name": "spmm_graph_large", "family": "spmm", "kind": "graph", "rows": 1000000, "mean": 16,
         "most": 10000, "n": 64, "dtype": "f32", "grad": True},
        # the same on a small graph with a narrow feature vector
        {"name": "spmm_graph_small", "family": "spmm", "kind": "graph", "rows": 20011, "mean": 5, "most": 170,
         "n": 16, "dtype": "f32", "grad": True},
        # A A on a volume grid with gradients of A's values
        {"name": "spgemm_grid3d", "family": "spgemm", "kind": "grid3d", "nx": 128, "ny": 128, "nz": 128,
         "dtype": "f64", "grad": True},
        # the two-hop graph A A of a graph with long rows
        {"name": "spgemm_graph", "family": "spgemm", "kind": "graph", "rows": 150000, "mean": 8, "most": 1000,
         "dtype": "f32", "grad": True},
        # the coarse-grid operator P^T A P of a learned interpolation, applied to a test vector, training
        {"name": "galerkin_grid2d", "family": "galerkin", "kind": "grid2d", "nx": 513, "ny": 641,
         "dtype": "f64", "grad": True},
        # symmetric part of a matrix (A + A^T) / 2, training
        {"name": "symmetric_part_grid2d", "family": "sum", "kind": "grid2d", "nx": 1201, "ny": 997,
         "dtype": "f32", "grad": True},
        # forward substitution and its adjoint on a plane grid (many short levels)
        {"name": "sptrsv_grid2d", "family": "sptrsv", "kind": "grid2d", "nx": 1024, "ny": 1024, "lower": True,
         "dtype": "f64", "grad": True},
        # backward substitution of a preconditioner on a volume grid (fewer, wider levels), no gradients
        {"name": "sptrsv_grid3d_apply", "family": "sptrsv", "kind": "grid3d", "nx": 97, "ny": 89, "nz": 101,
         "lower": False, "dtype": "f32", "grad": False},
        # a direct solve and its gradients
        {"name": "spsolve_grid2d", "family": "spsolve", "kind": "grid2d", "nx": 64, "ny": 64, "dtype": "f64",
         "grad": True},
    ]


def _size(rng, low, high):
    """Between low and high, spread evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _grid2d(rng, low, high):
    return {"kind": "grid2d", "nx": _size(rng, low, high), "ny": _size(rng, low, high)}


def _grid3d(rng, low, high):
    return {"kind": "grid3d", "nx": _size(rng, low, high), "ny": _size(rng, low, high), "nz": _size(rng, low, high)}


def _graph(rng, low, high, mean, most):
    return {"kind": "graph", "rows": _size(rng, low, high), "mean": rng.randint(3, mean), "most": _size(rng, 100, most)}


def draw(rng):
    family = rng.choice(["spmv", "spmv", "spmm", "spmm", "spgemm", "spgemm", "galerkin", "sum", "sptrsv", "sptrsv",
                         "spsolve"])
    case = {"family": family}
    dtype, grad = rng.choice(["f32", "f64"]), True
    if family == "spmv":
        case.update(rng.choice([_grid2d(rng, 100, 2000), _grid3d(rng, 20, 150), _graph(rng, 4000, 400000, 20, 5000)]))
        grad = rng.random() < 0.6
    elif family == "spmm":
        if rng.random() < 0.6:
            case.update(_graph(rng, 3000, 1000000, 16, 10000))
            # feature widths; the widest ones belong to the smaller graphs
            case["n"] = min(_size(rng, 8, 128), max(8, int(1e9 / (case["rows"] * case["mean"]))))
            dtype = rng.choice(["f32", "f32", "f64"])
        else:
            # a block of right-hand sides
            case.update(_grid3d(rng, 16, 96))
            case["n"] = _size(rng, 2, 16)
        grad = rng.random() < 0.7
        if case["n"] > 64 and dtype == "f64":
            dtype = "f32"
    elif family == "spgemm":
        case.update(rng.choice([_grid2d(rng, 60, 1000), _grid3d(rng, 16, 120), _graph(rng, 5000, 140000, 8, 1000)]))
        grad = rng.random() < 0.7
    elif family == "galerkin":
        case.update(_grid2d(rng, 50, 640))
    elif family == "sum":
        case.update(_grid2d(rng, 60, 1100))
    elif family == "sptrsv":
        if rng.random() < 0.5:
            case.update(_grid2d(rng, 60, 1000))
        else:
            case.update(_grid3d(rng, 16, 96))
        case["lower"] = rng.random() < 0.5
        grad = rng.random() < 0.6
    else:
        case.update(_grid2d(rng, 12, 64))
        dtype = "f64"
    case.update({"dtype": dtype, "grad": grad})
    return case


# ---- inputs ------------------------------------------------------------------------

def _dims(case):
    return [case[k] for k in ("nx", "ny", "nz") if k in case]


def _rows(case):
    return case["rows"] if case["kind"] == "graph" else math.prod(_dims(case))


def _assemble(columns, valid, values):
    """CSR arrays out of one row per grid point: its columns in ascending order, which of them
    exist, and the values."""
    indptr = torch.zeros(columns.shape[0] + 1, dtype=torch.int64, device="cuda")
    indptr[1:] = torch.cumsum(valid.sum(1), 0)
    return values[valid].contiguous(), columns[valid].contiguous(), indptr


def _stencil(case, gen, dtype, part="all"):
    """Five-point or seven-point matrix: twice the dimension on the diagonal, -1 off it, every
    value scaled by 1 + 0.01 U(-1, 1); a triangle of it has a diagonal larger by U(0, 1)."""
    dims = _dims(case)
    N, d = math.prod(dims), len(dims)
    r = torch.arange(N, device="cuda")
    below, above, stride = [], [], 1
    for n in reversed(dims):
        at = (r // stride) % n
        below.append((-stride, at > 0))
        above.append((stride, at < n - 1))
        stride *= n
    legs = list(reversed(below)) * (part != "upper") + [(0, None)] + above * (part != "lower")
    columns = torch.stack([r + off for off, _ in legs], 1)
    valid = torch.stack([torch.ones_like(r, dtype=torch.bool) if ok is None else ok for _, ok in legs], 1)
    noise = torch.rand(N, len(legs), generator=gen, device="cuda", dtype=torch.float64)
    values = torch.where(columns == r[:, None], 2.0 * d, -1.0).double() * (1.0 + 0.01 * (2.0 * noise - 1.0))
    if part != "all":
        on = torch.arange(N, device="cuda")
        at = [off for off, _ in legs].index(0)
        values[on, at] = 2.0 * d + noise[:, at]
    return _assemble(columns, valid, values.to(dtype))


def _power_law(case, gen, dtype):
    """Graph with degrees of tail exponent 2.1 and about the given mean, none above `most`, dealt to the
    rows at random; each of a row's columns is uniformly random in its own share of all columns,
    values U(0, 2) over the row's degree."""
    rows = case["rows"]
    u = (torch.arange(rows, device="cuda", dtype=torch.float64) + 0.5) / rows
    degree = torch.floor(u ** (-1.0 / 1.1)).clamp_max(case["most"])
    degree = torch.ceil(degree * (case["mean"] * rows / degree.sum())).clamp(1, min(case["most"], rows // 2)).long()
    # the entries of a product of such patterns depend on the draw: its graph is the same for every
    # seed, only the values change
    shape = gen
    if case["family"] == "spgemm":
        shape = torch.Generator(device="cuda")
        shape.manual_seed(rows)
    degree = degree[torch.randperm(rows, generator=shape, device="cuda")]
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    indptr[1:] = torch.cumsum(degree, 0)
    row = torch.repeat_interleave(torch.arange(rows, device="cuda"), degree)
    k, d = torch.arange(row.numel(), device="cuda") - indptr[row], degree[row]
    low, high = k * rows // d, (k + 1) * rows // d
    at = torch.rand(row.numel(), generator=shape, device="cuda", dtype=torch.float64)
    columns = torch.minimum(low + (at * (high - low)).long(), high - 1)
    values = 2.0 * torch.rand(row.numel(), generator=gen, device="cuda", dtype=torch.float64) / d
    return values.to(dtype), columns, indptr


def _interpolation(case, gen, dtype):
    """Bilinear interpolation from every second grid line, weights scaled by 1 + 0.01 U(-1, 1)."""
    nx, ny = case["nx"], case["ny"]
    cx, cy = (nx + 1) // 2, (ny + 1) // 2
    r = torch.arange(nx * ny, device="cuda")
    i, j = r // ny, r % ny
    legs = []
    for di in (0, 1):
        for dj in (0, 1):
            I, J = i // 2 + di, j // 2 + dj
            ok = (I < cx) & (J < cy) & ((di == 0) | (i % 2 == 1)) & ((dj == 0) | (j % 2 == 1))
            w = torch.where(i % 2 == 1, 0.5, 1.0) * torch.where(j % 2 == 1, 0.5, 1.0)
            legs.append((I * cy + J, ok, w.double()))
    noise = torch.rand(r.numel(), 4, generator=gen, device="cuda", dtype=torch.float64)
    values = torch.stack([w for _, _, w in legs], 1) * (1.0 + 0.01 * (2.0 * noise - 1.0))
    arrays = _assemble(torch.stack([c for c, _, _ in legs], 1), torch.stack([ok for _, ok, _ in legs], 1),
                       values.to(dtype))
    return arrays, (nx * ny, cx * cy)


def _product_bound(A):
    """More entries than A A can have."""
    lengths = A.indptr[1:] - A.indptr[:-1]
    return int(lengths[A.indices].sum())


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype, grad, family = DTYPES[case["dtype"]], case["grad"], case["family"]
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)  # noqa: E731
    rows = _rows(case)
    if case["kind"] == "graph":
        arrays = _power_law(case, gen, dtype)
    else:
        part = "all" if family != "sptrsv" else "lower" if case["lower"] else "upper"
        arrays = _stencil(case, gen, dtype, part)
    A = sp.SparseCSRTensor(arrays, (rows, rows), clone=False)
    A.requires_grad = grad
    state = {"case": case, "A": A}
    if family in ("spmv", "sptrsv", "spsolve"):
        state["x"] = normal(rows).requires_grad_(grad)
        state["g"] = normal(rows)
    elif family == "spmm":
        state["x"] = normal(rows, case["n"]).requires_grad_(grad)
        state["g"] = normal(rows, case["n"])
    elif family == "spgemm":
        # the gradient that comes back on the product's entries: as many of these as it has
        state["g"] = normal(_product_bound(A)) if grad and case["kind"] == "graph" else \
            normal(_nnz_of_square(case)) if grad else None
    elif family == "sum":
        state["g"] = normal(A.nnz)
    elif family == "galerkin":
        P, shape = _interpolation(case, gen, dtype)
        state["P"] = sp.SparseCSRTensor(P, shape, clone=False)
        state["P"].requires_grad = True
        state["x"], state["g"] = normal(shape[1]), normal(shape[1])
    return state


# ---- one pass ----------------------------------------------------------------------

def run(state):
    case, A = state["case"], state["A"]
    family, grad = case["family"], case["grad"]
    x, g = state.get("x"), state.get("g")
    if family == "spmv" or family == "spmm":
        y = A @ x
        return (y,) + torch.autograd.grad(y, (A.data, x), g) if grad else y
    if family == "sptrsv":
        y = linalg.spsolve_triangular(A, x, lower=case["lower"])
        return (y,) + torch.autograd.grad(y, (A.data, x), g) if grad else y
    if family == "spsolve":
        y = linalg.spsolve(A, x)
        return (y,) + torch.autograd.grad(y, (A.data, x), g)
    if family == "spgemm":
        C = A @ A
        out = (C.data, C.indices, C.indptr)
        return out + torch.autograd.grad(C.data, A.data, g[:C.nnz]) if grad else out
    if family == "sum":
        C = (A + A.T) * 0.5
        return (C.data, C.indices, C.indptr) + torch.autograd.grad(C.data, A.data, g)
    P = state["P"]
    C = P.T @ (A @ P)
    y = C @ x
    return (C.data, C.indices, C.indptr, y) + torch.autograd.grad(y, (A.data, P.data), g)


# ---- what a pass cannot do without -------------------------------------------------

def _nnz(case):
    if case["kind"] == "graph":
        return case["rows"] * case["mean"]
    dims = _dims(case)
    N = math.prod(dims)
    off = sum(N // n * (n - 1) for n in dims)
    return N + off * (1 if case["family"] == "sptrsv" else 2)


def _nnz_of_square(case):
    """Entries of A A: every sum of two steps of the stencil that stays on the grid."""
    if case["kind"] == "graph":
        return int(case["rows"] * case["mean"] ** 2 * 0.98)
    dims = _dims(case)
    steps = {tuple(0 for _ in dims)}
    for k in range(len(dims)):
        for s in (-1, 1):
            steps.add(tuple(s if j == k else 0 for j in range(len(dims))))
    both = {tuple(a + b for a, b in zip(p, q)) for p in steps for q in steps}
    return sum(math.prod(max(n - abs(o), 0) for n, o in zip(dims, step)) for step in both)


def work(case):
    """Values and vectors at their width, the structure of the operands at 32 bits, the structure
    of a result at 64: each read or written once, forward and (where gradients are asked for) backward."""
    s = 4 if case["dtype"] == "f32" else 8
    family, grad = case["family"], case["grad"]
    N, nnz = _rows(case), _nnz(case)
    structure = 4 * (nnz + N + 1)
    if family in ("spmv", "spmm"):
        n = case.get("n", 1)
        dense = N * n * s
        return {"bytes": structure + nnz * s + 2 * dense + (structure + 2 * nnz * s + 3 * dense if grad else 0),
                "flops": 2 * nnz * n * (3 if grad else 1)}
    if family == "sptrsv":
        return {"bytes": structure + nnz * s + 2 * N * s + (structure + 2 * nnz * s + 3 * N * s if grad else 0),
                "flops": 2 * nnz + (3 * nnz if grad else 0)}
    if family == "spsolve":
        # the factors of a band as wide as the grid's lines are neither input nor result: operations only
        fill = N * (2 * case["ny"] + 1)
        return {"bytes": 2 * structure + nnz * (3 * s) + 5 * N * s, "flops": 2 * N * case["ny"] ** 2 + 8 * fill}
    if family == "spgemm":
        C = _nnz_of_square(case)
        products = case["rows"] * case["mean"] ** 2 if case["kind"] == "graph" else nnz * nnz // N
        return {"bytes": structure + nnz * s + C * (s + 8) + 8 * N +
                (structure + C * s + 2 * nnz * s if grad else 0), "flops": 2 * products * (3 if grad else 1)}
    if family == "sum":
        return {"bytes": structure + nnz * (s + s + 8) + 8 * N + structure + 2 * nnz * s, "flops": 6 * nnz}
    pn, cn = 9 * N // 4, N // 4
    C = 9 * cn
    return {"bytes": structure + nnz * s + pn * (s + 4) + C * (s + 8) + 8 * cn + 3 * cn * s +
            structure + 2 * nnz * s + 2 * pn * s, "flops": 3 * 2 * (nnz * 9 // 4 + pn * 5 + C)}


def tolerance(case):
    """About four times what the 32-bit path differs from the same inputs in 64 bits (largest seen: 1.2e-7
    and 1.9e-6, the coarse-grid operator; direct solves, 3e-4 and 5.3e-4), and that over 2^29 for 64-bit
    values."""
    if case["family"] == "spsolve":
        return {"rel": 2.5e-12, "max": 4e-12}
    return {"rel": 5e-7, "max": 8e-6} if case["dtype"] == "f32" else {"rel": 1e-15, "max": 1.5e-14}
