"""Stretches of wide levels, which one launch takes row by row (sptrsv_flow_kernel): the serial loop's
results bit for bit, whichever way the levels go."""
import numpy as np
import pytest
import torch

import numml_amd
import oracle
from numml_amd import _lib
from util import assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


def _grid(dims, dtype, lower, seed):
    """Triangle of a stencil on a grid of any dimension, but for one coupling (else a plane's or volume's is solved line
    by line and not here)."""
    n = int(np.prod(dims))
    r = np.arange(n)
    stride, rows, cols = 1, [r], [r]
    for d in reversed(dims):
        ok = (r // stride) % d > 0
        rows.append(r[ok])
        cols.append(r[ok] - stride)
        stride *= d
    r, c = np.concatenate(rows), np.concatenate(cols)
    keep = (r != n // 2 + 1) | (c != n // 2)
    assert not keep.all()
    r, c = r[keep], c[keep]
    if not lower:
        r, c = c, r
    return _csr(r, c, n, dtype, seed)


def _layers(width, layers, deps, dtype, lower, seed):
    """`layers` levels of `width` rows; a row depends on one row of the layer before and on up to
    deps - 1 rows of any earlier layer."""
    rng = np.random.default_rng(seed)
    n = width * layers
    r, c = [np.arange(n)], [np.arange(n)]
    at = np.arange(width, n)
    layer = at // width
    r.append(at)
    c.append((layer - 1) * width + rng.integers(0, width, at.size))
    for _ in range(deps - 1):
        r.append(at)
        c.append((rng.random(at.size) * layer * width).astype(np.int64))
    r, c = np.concatenate(r), np.concatenate(c)
    rc = np.unique(np.stack([r, c], 1), axis=0)
    r, c = rc[:, 0], rc[:, 1]
    if not lower:
        r, c = n - 1 - r, n - 1 - c
    return _csr(r, c, n, dtype, seed)


def _csr(r, c, n, dtype, seed):
    rng = np.random.default_rng(seed)
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    d = rng.uniform(-1, 1, r.size) * 0.3
    d[r == c] = rng.uniform(1, 2, n)
    p = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(r, minlength=n), out=p[1:])
    return d.astype(dtype), c.astype(np.int64), p, n


def _compare(dev, d, i, p, n, dtype, lower, unit, b=None):
    ext = numml_amd.load_compiled()
    b = randn(5, n, dtype) if b is None else b
    g = randn(6, n, dtype)
    D, I, P, Bv, Gv = to_dev(dev, d, i, p, b, g)
    x_ref = oracle.sptrsv_forward(n, n, d, i, p, lower, unit, b)
    for one_workgroup in (0, 2):
        try:
            assert _lib.lib().nm_sptrsv_configure(0, one_workgroup) == 0
            x = ext.sptrsv_forward(n, n, D, I, P, lower, unit, Bv)
            grads = ext.sptrsv_backward(Gv, x, n, n, D, I, P, lower, unit, Bv)
        finally:
            assert _lib.lib().nm_sptrsv_configure(0, 0) == 0
        assert_same(host(x), x_ref, f"x, bits {one_workgroup}")
        for got, ref in zip(grads, oracle.sptrsv_backward(g, x_ref, n, n, d, i, p, lower, unit, b)):
            assert_same(host(got), ref, f"gradient, bits {one_workgroup}")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims, lower, unit", [((40, 41, 43), True, False), ((61, 47, 50), False, False),
                                               ((9, 10, 11, 12, 13), True, True), ((70, 64, 33), True, True)])
def test_grids(dev, dtype, dims, lower, unit):
    print("case", dims, dtype.__name__, flush=True)
    d, i, p, n = _grid(dims, dtype, lower, 1)
    _compare(dev, d, i, p, n, dtype, lower, unit)
    ext = numml_amd.load_compiled()
    I, P = to_dev(dev, i, p)
    one = ext.sptrsv_schedule(n, I, P, lower)[1]
    try:
        assert _lib.lib().nm_sptrsv_configure(0, 2) == 0
        assert 1 < one < ext.sptrsv_schedule(n, I, P, lower)[1] - 4   # the wide levels one by one, the narrow ones elsewhere
    finally:
        assert _lib.lib().nm_sptrsv_configure(0, 0) == 0


# layers at the edges of what goes level by level (1024 rows, 2 levels), of tiles (64 rows) and of the
# operand widths (2, 4, 8 dependencies; 9 take the other way)
@pytest.mark.parametrize("width, layers, deps", [(1025, 4, 1), (1025, 3, 2), (1025, 2, 1), (30000, 2, 4),
                                                 (40000, 4, 8), (1087, 9, 2), (4097, 6, 3), (5000, 5, 4),
                                                 (1100, 12, 5), (6001, 7, 8), (4200, 6, 9), (70000, 5, 3), (1500, 40, 4)])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_layers(dev, width, layers, deps, lower, dtype):
    print("case", width, layers, deps, lower, dtype.__name__, flush=True)
    d, i, p, n = _layers(width, layers, deps, dtype, lower, width)
    _compare(dev, d, i, p, n, dtype, lower, False)
    # one launch for all the layers, which is what gives up where waiting is not allowed
    ext = numml_amd.load_compiled()
    D, I, P, Bv = to_dev(dev, d, i, p, randn(5, n, dtype))
    one = deps <= 8
    assert tuple(ext.sptrsv_schedule(n, I, P, lower)) == (layers, 1 if one else layers)
    try:
        assert _lib.lib().nm_sptrsv_configure(-1, 0) == 0
        assert bool(torch.isnan(ext.sptrsv_forward(n, n, D, I, P, lower, False, Bv)).all()) == one
    finally:
        assert _lib.lib().nm_sptrsv_configure(0, 0) == 0


def test_not_a_number_and_infinity(dev):
    # every NaN there is passes from row to row, the one that marks an unsolved row among them
    d, i, p, n = _grid((40, 41, 43), np.float64, True, 2)
    b = randn(7, n, np.float64)
    b[[50, 20000]] = np.inf
    b.view(np.uint64)[[0, 7000, 30000, 60000]] = 0xffffffffffffffff
    _compare(dev, d, i, p, n, np.float64, True, False, b)


def test_gives_up_instead_of_waiting_forever(dev):
    d, i, p, n = _layers(5000, 6, 3, np.float64, True, 3)
    D, I, P, Bv = to_dev(dev, d, i, p, randn(8, n, np.float64))
    ext = numml_amd.load_compiled()
    try:
        assert _lib.lib().nm_sptrsv_configure(-1, 0) == 0
        x = ext.sptrsv_forward(n, n, D, I, P, True, False, Bv)
        torch.cuda.synchronize()
        assert bool(torch.isnan(x).all())
    finally:
        assert _lib.lib().nm_sptrsv_configure(0, 0) == 0


def test_in_a_graph(dev):
    d, i, p, n = _grid((50, 41, 43), np.float64, True, 4)
    ext = numml_amd.load_compiled()
    D, I, P = to_dev(dev, d, i, p)
    b1, b2 = to_dev(dev, randn(9, n, np.float64), randn(10, n, np.float64))
    held = b1.clone()
    ext.sptrsv_forward(n, n, D, I, P, True, False, held)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x = ext.sptrsv_forward(n, n, D, I, P, True, False, held)
    for b in (b1, b2, b1, b2):
        held.copy_(b)
        graph.replay()
        want = ext.sptrsv_forward(n, n, D, I, P, True, False, b)
        torch.cuda.synchronize()
        assert torch.equal(x, want)


# one workgroup in two of such a launch starts when another has ended; the wavefronts that wait for its rows
# have to solve these themselves (dependencies of one row: 1, 3 and up to 8)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("deps, lower", [(1, True), (3, False), (8, True)])
def test_more_workgroups_than_run_at_once(dev, dtype, deps, lower):
    print("case", deps, lower, dtype.__name__, flush=True)
    d, i, p, n = _layers(20000, 20, deps, dtype, lower, deps)
    b, g = randn(5, n, dtype), randn(6, n, dtype)
    D, I, P, Bv, Gv = to_dev(dev, d, i, p, b, g)
    x_ref = oracle.sptrsv_forward(n, n, d, i, p, lower, False, b)
    ext = numml_amd.load_compiled()
    try:
        assert _lib.lib().nm_sptrsv_configure(0, 4) == 0
        x = ext.sptrsv_forward(n, n, D, I, P, lower, False, Bv)
        grads = ext.sptrsv_backward(Gv, x, n, n, D, I, P, lower, False, Bv)
        torch.cuda.synchronize()
    finally:
        assert _lib.lib().nm_sptrsv_configure(0, 0) == 0
    assert_same(host(x), x_ref, "x")
    for got, ref in zip(grads, oracle.sptrsv_backward(g, x_ref, n, n, d, i, p, lower, False, b)):
        assert_same(host(got), ref, "gradient")


def test_on_four_streams_at_once(dev):
    d, i, p, n = _layers(20000, 20, 8, np.float64, True, 11)
    ext = numml_amd.load_compiled()
    D, I, P = to_dev(dev, d, i, p)
    bs = to_dev(dev, *(randn(20 + k, n, np.float64) for k in range(4)))
    want = [ext.sptrsv_forward(n, n, D, I, P, True, False, b) for b in bs]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in bs], []
    for _ in range(3):
        for b, s in zip(bs, streams):
            with torch.cuda.stream(s):
                got.append(ext.sptrsv_forward(n, n, D, I, P, True, False, b))
    torch.cuda.synchronize()
    for k, x in enumerate(got):
        assert torch.equal(x, want[k % 4])
