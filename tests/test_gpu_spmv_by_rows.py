"""Gradients of matrix-vector products that are made by rows: the gradient of A alone, both with the products brought into
column-major order, and the sums that are added to memory; those made by columns in narrow tiles; at the edges of
quads, tiles and long rows, against the oracle; and the default mode's choice among them."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from numml_amd import _binding, _lib
from numml_amd import generators as G
from numml_amd import numml_torch_cpp as ext
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


def _lengths(*lens, cols):
    lens = np.concatenate([np.atleast_1d(n) for n in lens])
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rng = np.random.default_rng(int(p[-1]))
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lens]).astype(np.int64)
    return i, p, (lens.size, cols)


def _case(case):
    if case == "one entry":
        return _lengths(1, cols=1)
    if case.startswith("quads"):                                    # entries of a tile modulo four
        return _lengths([3] * 20, int(case[-1]), cols=9)
    if case == "long rows":                                         # around kLongRow, a tile, and above it
        return _lengths([2] * 70, 31, 32, 33, 4095, [0] * 5, 4096, 4097, [1] * 600, 9000, cols=9100)
    if case == "long rows of few":                                  # more than eight entries a row: small tiles
        return _lengths([40] * 30, 1023, [9] * 50, 1024, 1025, [12] * 7, 5000, cols=5100)
    if case == "one column":
        return _lengths([1] * 5000, cols=1)
    if case == "wide":
        return _lengths([7] * 300, cols=200_000)
    if "band" in case:
        reach = [0, 1, 2, 3, 4, 5] if case == "band" else [0, 1, 2, 90, 700, 1500, 3000]
        n = 3000 if case == "band" else 9001
        offs = np.array(sorted({-o for o in reach} | set(reach)))
        c = np.arange(n)[:, None] + offs
        ok = (c >= 0) & (c < n)
        if case == "uneven band":                                   # not a symmetric pattern
            ok[::7, :4] = False
        return c[ok].astype(np.int64), np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int64), (n, n)
    d, i, p, shape = {"scattered": lambda: G.random_csr(3000, 2000, 0.01, 5), "ragged": lambda: G.ragged_csr(4000, 1500, 31, 8),
                      "grid": lambda: G.poisson2d(70)}[case]()
    return i, p, shape


CASES = ["one entry", "quads 1", "quads 2", "quads 3", "quads 4", "long rows", "long rows of few", "one column", "wide",
         "scattered", "ragged", "grid", "band", "far band", "uneven band"]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", CASES)
def test_against_the_oracle(dev, dtype, case):
    i, p, (rows, cols) = _case(case)
    d, x, g = randn(1, i.size, dtype), randn(2, cols, dtype), randn(3, rows, dtype)
    if case == "scattered":
        x[5], g[7], d[100], d[200] = np.inf, np.nan, -np.inf, np.nan
    want_A, want_x = oracle.spgemv_backward(g, rows, cols, d, i, p, x)
    D, I, P, X, Gz = to_dev(dev, d, i, p, x, g)
    L, dt, nnz = _lib.lib(), ext._dt(D), d.size
    plan = ext._transpose_plan(I, P, rows, cols, dev)
    pb, wb, sb = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    assert L.nm_permute_plan_bytes(nnz, pb, wb) == 0 and L.nm_spgemv_staged_bytes(dt, nnz, sb) == 0
    perm, work, room = (torch.empty(b.value, dtype=torch.uint8, device=dev) for b in (pb, wb, sb))
    assert L.nm_permute_plan_build(rows, cols, nnz, plan.mem.data_ptr(), perm.data_ptr(), pb, work.data_ptr(), wb, None) == 0
    short = np.bincount(i, minlength=cols) < 32        # (a longer column may be shared by a wavefront)

    # sums of the same terms in another order differ by less than 2 n eps times the sum of their sizes
    terms = np.bincount(i, minlength=cols)
    with np.errstate(invalid="ignore"):
        size = np.bincount(i, weights=np.abs(d.astype(np.float64) * g[np.repeat(np.arange(rows), np.diff(p))]), minlength=cols)
    finite = np.isfinite(want_x)

    def assert_sums(got, what):
        err = np.abs(got[finite].astype(np.float64) - want_x[finite])
        assert (err <= 2 * terms[finite] * np.finfo(dtype).eps * size[finite]).all(), what
        assert np.array_equal(got[~finite], want_x[~finite], equal_nan=True), what

    def fresh():
        return torch.full_like(D, 7), torch.full_like(X, 7)
    vectors = (X.data_ptr(), Gz.data_ptr())
    staged = (dt, rows, cols, nnz, D.data_ptr(), plan.mem.data_ptr(), perm.data_ptr(), room.data_ptr())
    for both in (True, False):
        gA, gx = fresh()
        assert L.nm_spgemv_backward_staged(*staged, sb, *vectors, gA.data_ptr() if both else None, gx.data_ptr(), None) == 0
        if both:
            assert_same(host(gA), want_A, "grad_A, staged")
        assert_same(host(gx)[short], want_x[short], "grad_x, staged")
        assert_sums(host(gx), "grad_x, staged")
    for planned in (L.nm_spgemv_backward_planned, L.nm_spgemv_backward_planned_lists):
        gA, _ = fresh()
        assert planned(dt, rows, cols, nnz, D.data_ptr(), plan.mem.data_ptr(), *vectors, gA.data_ptr(), None, None) == 0
        assert_same(host(gA), want_A, "grad_A alone, on the plan")
        for both in (True, False):
            gA, gx = fresh()
            assert planned(dt, rows, cols, nnz, D.data_ptr(), plan.mem.data_ptr(), *vectors, gA.data_ptr() if both else None,
                           gx.data_ptr(), None) == 0
            if both:
                assert_same(host(gA), want_A, "grad_A, on the plan")
            assert_same(host(gx)[short], want_x[short], "grad_x, on the plan")
            assert_sums(host(gx), "grad_x, on the plan")
    for both in (True, False):
        gA, gx = fresh()
        assert L.nm_spgemv_backward(dt, rows, cols, nnz, D.data_ptr(), I.data_ptr(), P.data_ptr(), *vectors, gA.data_ptr(),
                                    gx.data_ptr() if both else None, None) == 0
        assert_same(host(gA), want_A, "grad_A, stateless")
        if both:
            assert_sums(host(gx), "grad_x, stateless")
    # memory that is too small and missing operands are refused
    assert L.nm_spgemv_backward_staged(*staged, sb.value - 1, *vectors, None, gx.data_ptr(), None) != 0
    assert L.nm_spgemv_backward_staged(*staged, sb, *vectors, gA.data_ptr(), None, None) != 0


@pytest.mark.skipif(_binding.name != "compiled", reason="the plan policy lives in the compiled binding")
def test_default_mode(dev):
    ops = _binding.ops
    old = ops.backward_mode()
    ops.set_backward_mode("planned")
    try:
        for case, plans_both, plans_x in (("scattered", 2, 1), ("grid", 1, 1)):
            ops.clear_plan_cache()
            if case == "grid":
                d, i, p, (rows, cols) = G.poisson2d(440, np.float32, jitter_seed=1)
            else:
                rows = cols = 200_000
                rng = np.random.default_rng(3)
                i = np.sort(rng.integers(0, cols, (rows, 5)), 1).reshape(-1)
                p, d = np.arange(rows + 1, dtype=np.int64) * 5, randn(1, 5 * rows, np.float32)
            D, I, P, X, Gz = to_dev(dev, d, i, p, randn(2, cols, np.float32), randn(3, rows, np.float32))
            want = oracle.spgemv_backward(host(Gz), rows, cols, d, i, p, host(X))
            for wants, held in (((False, True), plans_x), ((True, False), plans_x), ((True, True), plans_both)):
                a, b = (t.clone().requires_grad_(w) for t, w in zip((D, X), wants))
                for _ in range(4):
                    out = ops.spgemv_backward(Gz, rows, cols, a, I, P, b)
                    for o, ref, w in zip(out, want, wants):
                        assert (o is None) != w
                        if w:
                            assert_close(host(o), ref, case)
                assert ops.plan_cache_size() == held, (case, wants)
            graph = torch.cuda.CUDAGraph()
            a, b = D.clone().requires_grad_(), X.clone().requires_grad_()
            torch.cuda.synchronize()
            with torch.cuda.graph(graph):
                out = ops.spgemv_backward(Gz, rows, cols, a, I, P, b)
            for k in range(3):
                Gz.copy_(torch.from_numpy(randn(20 + k, rows, np.float32)))
                graph.replay()
                torch.cuda.synchronize()
                now = ops.spgemv_backward(Gz, rows, cols, a, I, P, b)
                assert torch.equal(out[0], now[0]) and torch.equal(out[1], now[1])
    finally:
        ops.set_backward_mode(old)
        ops.clear_plan_cache()


def _spread_rows(rows, at, lens):
    n = np.zeros(rows, np.int64)
    n[at] = lens
    return n


TILES = {   # lengths of the rows; a workgroup of the kernel by entries stages 1024 rows at a time, up to 4096 of them
    "one row": np.array([70_000]),
    "ends of tiles": np.array([255, 1, 256, 257, 511, 64, 63, 1, 1, 128, 2]),
    "all empty but one": _spread_rows(100_000, [99_000], [3]),
    "empty ones first and last": _spread_rows(20_000, [9_000, 9_001], [300, 5]),
    "1023 to 1025 rows a tile": np.concatenate([_spread_rows(1022, [0, 500], [100, 156]), _spread_rows(1024, [1023], [256]),
                                                _spread_rows(1025, [3, 1024], [1, 255]), [300]]),
    "4095 to 4097 rows a tile": np.concatenate([_spread_rows(4094, [0, 500], [100, 156]), _spread_rows(4096, [4095], [256]),
                                                _spread_rows(4098, [3, 4097], [1, 255]), [300]]),
    "many entries": np.concatenate([np.full(500_000, 3), [600_000], np.zeros(9000, np.int64), [1, 2047, 2048, 2049], np.full(3000, 40), [17]]),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", list(TILES))
def test_gradient_of_the_matrix_alone_on_the_plan(dev, dtype, case):
    lens, cols = TILES[case], 1000
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rows, nnz = lens.size, int(p[-1])
    i = np.random.default_rng(nnz).integers(0, cols, nnz)
    d, x, g = randn(1, nnz, dtype), randn(2, cols, dtype), randn(3, rows, dtype)
    X, Gz = to_dev(dev, x, g)
    L, dt = _lib.lib(), ext._dt(X)
    for n in (nnz, nnz - 1, nnz - 63) if lens[-1] > 63 else (nnz,):      # other ends of the last tile
        p[-1] = n
        D, I, P = to_dev(dev, d[:n], i[:n], p)
        plan = ext._transpose_plan(I, P, rows, cols, dev)
        out = torch.full((n + 8,), 7, dtype=D.dtype, device=dev)
        assert L.nm_spgemv_backward_planned(dt, rows, cols, n, D.data_ptr(), plan.mem.data_ptr(), X.data_ptr(), Gz.data_ptr(),
                                            out.data_ptr(), None, None) == 0
        want = g[np.repeat(np.arange(rows), np.diff(p))] * x[i[:n]]
        assert_same(host(out)[:n], want, f"{case}, {n} entries")
        assert (host(out)[n:] == 7).all()
        # the products of the way through column-major order are made by the same kernel
        pb, wb, sb = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
        assert L.nm_permute_plan_bytes(n, pb, wb) == 0 and L.nm_spgemv_staged_bytes(dt, n, sb) == 0
        perm, work, room = (torch.empty(b.value, dtype=torch.uint8, device=dev) for b in (pb, wb, sb))
        assert L.nm_permute_plan_build(rows, cols, n, plan.mem.data_ptr(), perm.data_ptr(), pb, work.data_ptr(), wb, None) == 0
        gA, gx = torch.empty_like(D), torch.empty_like(X)
        assert L.nm_spgemv_backward_staged(dt, rows, cols, n, D.data_ptr(), plan.mem.data_ptr(), perm.data_ptr(), room.data_ptr(), sb,
                                           X.data_ptr(), Gz.data_ptr(), gA.data_ptr(), gx.data_ptr(), None) == 0
        assert_same(host(gA), want, f"{case}, {n} entries, with the gradient of x")
        terms = np.abs(g[np.repeat(np.arange(rows), np.diff(p))] * d[:n]).astype(np.float64)
        ref = np.bincount(i[:n], weights=(g[np.repeat(np.arange(rows), np.diff(p))] * d[:n]).astype(np.float64), minlength=cols)
        # sums of n terms in any order: 2 n eps times the sum of their sizes
        bound = 2 * np.finfo(dtype).eps * np.bincount(i[:n], minlength=cols) * np.bincount(i[:n], weights=terms, minlength=cols)
        assert (np.abs(host(gx) - ref) <= bound + 1e-300).all(), f"{case}: gradient of x"
