"""Triangles of five-point and seven-point matrices, which are solved line by line (nm_sptrsv_lines.hpp): the serial
loop's bits, forward and backward, at the edges of lines, patches and blocks of steps, and whatever the values."""
import numpy as np
import pytest
import torch

import numml_amd
import oracle
from numml_amd import _lib
from util import assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


def _triangle(dims, lower, seed, whole=False):
    """CSR triangle of a stencil on a grid (`whole`: with the other half of the matrix, which a solve passes over)."""
    rng = np.random.default_rng(seed)
    n = int(np.prod(dims))
    at = np.arange(n)
    stride, rows, cols = 1, [at], [at]
    for d in reversed(dims):
        ok = at // stride % d > 0
        for a, b in ((at[ok], at[ok] - stride), (at[ok] - stride, at[ok])):
            if whole or (b < a).all() == lower or a.size == 0:
                rows.append(a)
                cols.append(b)
        stride *= d
    r, c = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    v = rng.uniform(-1, 1, r.size) * 0.4
    v[r == c] = rng.uniform(1, 2, n)
    p = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(r, minlength=n), out=p[1:])
    return v, c.astype(np.int64), p, n


def _compare(dev, d, i, p, n, dtype, lower, unit, b=None, by_lines=True):
    ext = numml_amd.load_compiled()
    d = d.astype(dtype)
    b = randn(5, n, dtype) if b is None else b.astype(dtype)
    g = randn(6, n, dtype)
    D, I, P, Bv, Gv = to_dev(dev, d, i, p, b, g)
    assert (ext.sptrsv_schedule(n, I, P, lower)[1] == 1) == by_lines
    with np.errstate(all="ignore"):
        x_ref = oracle.sptrsv_forward(n, n, d, i, p, lower, unit, b)
        refs = oracle.sptrsv_backward(g, x_ref, n, n, d, i, p, lower, unit, b)
    x = ext.sptrsv_forward(n, n, D, I, P, lower, unit, Bv)
    assert_same(host(x), x_ref, "x")
    for got, ref, what in zip(ext.sptrsv_backward(Gv, x, n, n, D, I, P, lower, unit, Bv), refs, ("grad_A", "grad_b")):
        assert_same(host(got), ref, what)


# widths around a wavefront's 64 lines, lengths around a block's 8 and 16 steps; volumes around 8 x 8 patches; the
# longest side in every place
DIMS = [(2, 3), (3, 2), (64, 2), (65, 2), (63, 7), (64, 8), (65, 9), (128, 15), (129, 16), (130, 17), (200, 65), (70, 150),
        (300, 301), (2, 2, 2), (3, 2, 5), (8, 8, 4), (9, 8, 8), (8, 9, 16), (17, 2, 33), (2, 40, 9), (16, 24, 17),
        (25, 31, 40), (33, 3, 70), (150, 40), (700, 9), (70, 9, 10), (10, 70, 9), (9, 80, 17), (90, 17, 18)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lower, unit", [(True, False), (False, False), (True, True)])
@pytest.mark.parametrize("dims", DIMS)
def test_grids(dev, dims, lower, unit, dtype):
    print("case", dims, lower, unit, dtype.__name__, flush=True)
    d, i, p, n = _triangle(dims, lower, sum(dims))
    _compare(dev, d, i, p, n, dtype, lower, unit)


@pytest.mark.parametrize("dims", [(70, 33), (10, 11, 12)])
@pytest.mark.parametrize("lower", [True, False])
def test_the_other_half_is_passed_over(dev, dims, lower):
    d, i, p, n = _triangle(dims, lower, 3, whole=True)
    _compare(dev, d, i, p, n, np.float64, lower, False)


@pytest.mark.parametrize("dims", [(70, 33), (10, 11, 12)])
def test_values_that_the_short_division_does_not_take(dev, dims):
    d, i, p, n = _triangle(dims, True, 4)
    row = np.repeat(np.arange(n), np.diff(p))
    diag = np.flatnonzero(row == i)
    rng = np.random.default_rng(4)
    d[diag[rng.choice(n, 40, False)]] *= 10.0 ** rng.integers(-300, 300, 40)
    for zeros, special in ((True, ()), (False, (np.inf,)), (False, (np.nan, -np.inf))):
        b = randn(7, n, np.float64) * 10.0 ** rng.integers(-200, 200, n)
        if zeros:
            b[rng.random(n) < 0.7] = 0.
            b[rng.random(n) < 0.2] = -0.
        for v in special:
            b[rng.choice(n, 3, False)] = v
        _compare(dev, d, i, p, n, np.float64, True, False, b)
    d[diag[n // 2]] = 0.
    _compare(dev, d, i, p, n, np.float64, True, False)
    b = randn(8, n, np.float64)
    b.view(np.uint64)[[0, n // 3, n - 1]] = 0xffffffffffffffff   # the bits that mark a row as not solved
    _compare(dev, d, i, p, n, np.float64, True, False, b)


@pytest.mark.parametrize("what", ["missing", "extra", "far", "diagonal"])
def test_patterns_that_are_almost_a_grids(dev, what):
    d, i, p, n = _triangle((300, 200), True, 5)
    row = np.repeat(np.arange(n), np.diff(p))
    keep = np.ones(d.size, bool)
    add = []
    if what == "missing":
        keep[np.flatnonzero((row == 777) & (i == 776))] = False
    elif what == "extra":
        add = [(1333, 1333 - 200 - 1)]
    elif what == "far":
        add = [(1900, 3)]
    else:
        keep[np.flatnonzero((row == 1234) & (i == 1234))] = False   # an infinity from there on, but a grid's triangle
    r = np.concatenate([row[keep], np.array([a for a, _ in add], np.int64)])
    c = np.concatenate([i[keep], np.array([b for _, b in add], np.int64)])
    v = np.concatenate([d[keep], np.full(len(add), 0.25)])
    order = np.lexsort((c, r))
    p = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(r, minlength=n), out=p[1:])
    _compare(dev, v[order], c[order], p, n, np.float64, True, False, by_lines=what == "diagonal")


def test_gives_up_instead_of_waiting_forever(dev):
    ext = numml_amd.load_compiled()
    for dims in ((300, 70), (20, 21, 22)):
        d, i, p, n = _triangle(dims, True, 6)
        D, I, P, Bv = to_dev(dev, d, i, p, randn(8, n, np.float64))
        try:
            assert _lib.lib().nm_sptrsv_configure(-1, 0) == 0
            x = ext.sptrsv_forward(n, n, D, I, P, True, False, Bv)
            torch.cuda.synchronize()
            assert bool(torch.isnan(x).all())
        finally:
            assert _lib.lib().nm_sptrsv_configure(0, 0) == 0
        _compare(dev, d, i, p, n, np.float64, True, False)


@pytest.mark.parametrize("dims", [(300, 70), (20, 21, 22)])
def test_in_a_graph_and_on_four_streams(dev, dims):
    ext = numml_amd.load_compiled()
    d, i, p, n = _triangle(dims, False, 7)
    D, I, P = to_dev(dev, d, i, p)
    bs = to_dev(dev, *(randn(20 + k, n, np.float64) for k in range(4)))
    want = [ext.sptrsv_forward(n, n, D, I, P, False, False, b) for b in bs]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in bs], []
    for _ in range(3):
        for b, s in zip(bs, streams):
            with torch.cuda.stream(s):
                got.append(ext.sptrsv_forward(n, n, D, I, P, False, False, b))
    torch.cuda.synchronize()
    for k, x in enumerate(got):
        assert torch.equal(x, want[k % 4])
    held = bs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x = ext.sptrsv_forward(n, n, D, I, P, False, False, held)
    for k in (1, 2, 0, 3):
        held.copy_(bs[k])
        graph.replay()
        eager = ext.sptrsv_forward(n, n, D, I, P, False, False, bs[(k + 1) % 4])
        torch.cuda.synchronize()
        assert torch.equal(x, want[k]) and torch.equal(eager, want[(k + 1) % 4])
