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
    if by_lines:   # and by nothing else
        assert tuple(ext.sptrsv_shared_launches(n, I, P, lower)) == tuple(ext.sptrsv_chain_levels(n, I, P, lower)) == (0, 0)
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
@pytest.mark.parametrize("lower, unit", [(True, False), (False, False), (True, True), (False, True)])
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


# (lines along each of the directions)
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("dims", [(70, 33), (33, 70), (10, 11, 12), (10, 70, 9), (70, 9, 10)])
def test_values_that_the_short_division_does_not_take(dev, dims, lower):
    d, i, p, n = _triangle(dims, lower, 4)
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
        _compare(dev, d, i, p, n, np.float64, lower, False, b)
    d[diag[n // 2]] = 0.
    _compare(dev, d, i, p, n, np.float64, lower, False)
    b = randn(8, n, np.float64)
    b.view(np.uint64)[[0, n // 3, n - 1]] = 0xffffffffffffffff   # the bits that mark a row as not solved
    _compare(dev, d, i, p, n, np.float64, lower, False, b)


@pytest.mark.parametrize("dims", [(70, 33), (10, 11, 12)])
@pytest.mark.parametrize("lower", [True, False])
def test_fp32_values_out_of_the_ordinary(dev, dims, lower):
    d, i, p, n = _triangle(dims, lower, 17)
    rng = np.random.default_rng(17)
    row = np.repeat(np.arange(n), np.diff(p))
    diag = np.flatnonzero(row == i)
    d[diag[rng.choice(n, 40, False)]] *= 10.0 ** rng.integers(-35, 35, 40)
    for special in ((), (np.inf,), (np.nan, -np.inf), (-0., 1e-44)):
        b = randn(18, n, np.float64) * 10.0 ** rng.integers(-30, 30, n)
        b[rng.random(n) < 0.3] = 0.
        for v in special:
            b[rng.choice(n, 3, False)] = v
        with np.errstate(all="ignore"):
            _compare(dev, d, i, p, n, np.float32, lower, False, b)
    d[diag[n // 2]] = 0.
    _compare(dev, d, i, p, n, np.float32, lower, False)


@pytest.mark.parametrize("dims", [(2, 40), (70, 33), (2, 2, 30), (10, 11, 12)])
@pytest.mark.parametrize("lower", [True, False])
def test_no_diagonal_stored(dev, dims, lower):
    d, i, p, n = _triangle(dims, lower, 19)
    row = np.repeat(np.arange(n), np.diff(p))
    keep = row != i
    p = np.concatenate(([0], np.cumsum(np.bincount(row[keep], minlength=n)))).astype(np.int64)
    for dtype in (np.float32, np.float64):
        _compare(dev, d[keep], i[keep], p, n, dtype, lower, True)


# lines along each direction, one patch and several, lines longer than sixteen blocks of eight steps
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims, lower", [((130, 400), True), ((400, 70), False), ((33, 9), True), ((9, 80, 300), False), ((300, 10, 11), True),
                                         ((10, 300, 17), True)])
def test_zeros_here_and_there(dev, dims, lower, dtype):
    # Half of the couplings are zero, so that a zero of the right-hand side makes a zero quotient: the wavefront changes to
    # divisions in full and back at any block, the first, the second of a round, the ramps at both ends.
    d, i, p, n = _triangle(dims, lower, 11)
    rng = np.random.default_rng(n)
    row = np.repeat(np.arange(n), np.diff(p))
    d[(row != i) & (rng.random(d.size) < 0.5)] = 0.
    for share in (2 / n, 30 / n, 0.01, 0.5):
        b = randn(12, n, np.float64)
        b[rng.random(n) < share] = 0.
        b[rng.random(n) < share / 4] = -0.
        _compare(dev, d, i, p, n, dtype, lower, False, b)


@pytest.mark.parametrize("dims, lower", [((70, 33), False), ((33, 70), True), ((10, 11, 12), False), ((9, 70, 10), True)])
def test_quotients_at_the_ends_of_the_short_division(dev, dims, lower):
    # diagonals around 2^+-128 and quotients around 2^+-800; decoupled rows, so that each has the quotient it is given
    d, i, p, n = _triangle(dims, lower, 13)
    rng = np.random.default_rng(13)
    row = np.repeat(np.arange(n), np.diff(p))
    d[row != i] = 0.
    for far in (790, 799, 801, 1010):
        e = rng.integers(-128, 128, n)
        d[row == i] = np.ldexp(rng.uniform(1, 2, n) * rng.choice([-1, 1], n), e)
        b = np.ldexp(rng.uniform(1, 2, n), np.clip(e + rng.choice([-far, far], n) + rng.integers(-2, 3, n), -1060, 1022))
        _compare(dev, d, i, p, n, np.float64, lower, False, b)


def _solve_time(solve):
    for _ in range(3):
        solve()
    best = np.inf
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            solve()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


@pytest.mark.parametrize("dims", [(300, 70), (64, 64), (20, 21, 22)])
def test_zeros_ahead_of_the_first_source_cost_little(dev, dims):
    # Measured 1.4, 1.2 and 1.1 times a dense right-hand side's time; 3.1, 2.4 and 2.0 when every block that has a zero was
    # made twice.
    ext = numml_amd.load_compiled()
    d, i, p, n = _triangle(dims, True, 14)
    D, I, P, dense = to_dev(dev, d, i, p, randn(15, n, np.float64))
    source = torch.zeros_like(dense)
    source[n - 1] = 1.
    t = [_solve_time(lambda: ext.sptrsv_forward(n, n, D, I, P, True, False, b)) for b in (dense, source)]
    assert t[1] < 1.75 * t[0], t


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


# what a workgroup does from its second patch on: a launch has a workgroup per patch up to 1024 of them, so without this only
# grids of 257^3 and more come to it
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims, lower, unit", [((300, 301), True, False), ((301, 150), False, True), ((25, 31, 40), True, False),
                                               ((33, 40, 18), False, False), ((20, 70, 21), True, True)])
def test_two_workgroups_take_all_patches(dev, dims, lower, unit, dtype):
    d, i, p, n = _triangle(dims, lower, 16)
    try:
        assert _lib.lib().nm_sptrsv_configure(0, 8) == 0
        _compare(dev, d, i, p, n, dtype, lower, unit)
        _compare(dev, d, i, p, n, dtype, lower, unit, np.where(np.arange(n) == n // 2, 1., 0.))
    finally:
        assert _lib.lib().nm_sptrsv_configure(0, 0) == 0


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
