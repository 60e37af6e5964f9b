"""Sparse times dense with several entries a request (nm_spmm_groups.hpp): dense operands around
every width at which the number of lanes an entry takes changes, and rows around the lengths from
which a workgroup shares them.  Against the serial oracle, bit for bit where its order is kept."""
import numpy as np
import pytest

import oracle
from numml_amd import numml_torch_cpp as ext
from util import assert_close, assert_same, randn, host, to_dev

pytestmark = pytest.mark.gpu


def _rows_of(lengths, cols, dtype, seed):
    rng = np.random.default_rng(seed)
    p = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lengths] + [[]]).astype(np.int64)
    return rng.standard_normal(i.size).astype(dtype), i, p, (len(lengths), cols)


# lengths around a chunk (16), the rows a workgroup shares (128) in storage order (512) and beyond
LENGTHS = [0, 1, 15, 16, 17, 0, 127, 128, 129, 2, 511, 512, 513, 3, 700, 1040, 0, 0, 5, 33]


@pytest.fixture(params=["eager", "atomic"])
def mode(request):
    old = ext.BACKWARD_MODE
    ext.BACKWARD_MODE = request.param
    yield request.param
    ext.BACKWARD_MODE = old


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 9, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 256, 257])
def test_widths_and_lengths(dev, dtype, n, mode):
    for name, lengths in (("edges", LENGTHS), ("short", [3] * 70), ("repeated", LENGTHS * 4)):
        d, i, p, (rows, cols) = _rows_of(lengths, 1100, dtype, 1)
        B, gC = randn(3, (cols, n), dtype), randn(4, (rows, n), dtype)
        D, I, P, Bd, Gd = to_dev(dev, d, i, p, B, gC)
        C, C_ref = host(ext.spdmm_forward(rows, cols, D, I, P, Bd)), oracle.spdmm_forward(rows, cols, d, i, p, B)
        kept = np.diff(p) <= 512
        assert_same(C[kept], C_ref[kept], f"{name} n={n} C, rows in storage order")
        assert_close(C, C_ref, f"{name} n={n} C")
        gA_ref, gB_ref = oracle.spdmm_backward(rows, cols, d, i, p, B, gC)
        gA, gB = ext.spdmm_backward(rows, cols, D, I, P, Bd, Gd)
        assert_close(host(gA), gA_ref, f"{name} n={n} grad_A")
        (assert_same if mode == "eager" else assert_close)(host(gB), gB_ref, f"{name} n={n} grad_B")
        Dr, Br = D.clone().requires_grad_(True), Bd.clone().requires_grad_(True)
        assert_close(host(ext.spdmm_backward(rows, cols, Dr, I, P, Bd, Gd)[0]), gA_ref, f"{name} n={n} grad_A alone")
        alone = host(ext.spdmm_backward(rows, cols, D, I, P, Br, Gd)[1])
        (assert_same if mode == "eager" else assert_close)(alone, gB_ref, f"{name} n={n} grad_B alone")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_long_columns_and_rows_off_alignment(dev, dtype):
    """The transpose's long columns in the backward; operands whose rows begin anywhere."""
    d, i, p, (rows, cols) = _rows_of(LENGTHS, 1100, dtype, 5)
    t = oracle.csr_transpose(rows, cols, d, i, p)
    d, i, p = t[0], t[1], t[2]
    rows, cols = cols, rows
    old, ext.BACKWARD_MODE = ext.BACKWARD_MODE, "eager"
    try:
        for n in (5, 30, 62, 100):
            B, gC = randn(6, (cols, n + 3), dtype), randn(7, (rows, n + 2), dtype)
            D, I, P, Bw, Gw = to_dev(dev, d, i, p, B, gC)
            Bd, Gd = Bw[:, 3:], Gw[:, 1:n + 1]
            C_ref = oracle.spdmm_forward(rows, cols, d, i, p, np.ascontiguousarray(B[:, 3:]))
            assert_same(host(ext.spdmm_forward(rows, cols, D, I, P, Bd)), C_ref, f"n={n} C")
            gA_ref, gB_ref = oracle.spdmm_backward(rows, cols, d, i, p, np.ascontiguousarray(B[:, 3:]),
                                                   np.ascontiguousarray(gC[:, 1:n + 1]))
            gA, gB = (host(v) for v in ext.spdmm_backward(rows, cols, D, I, P, Bd, Gd))
            assert_close(gA, gA_ref, f"n={n} grad_A")
            assert_close(gB, gB_ref, f"n={n} grad_B")
            kept = np.bincount(i, minlength=cols) <= 512
            assert_same(gB[kept], gB_ref[kept], f"n={n} grad_B, columns in storage order")
    finally:
        ext.BACKWARD_MODE = old


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 2500, 40_000, 140_000, 300_001, 600_001])
def test_long_rows_side_by_side(dev, dtype, rows, mode):
    """Blocks of long rows among short ones, where the rows are dealt to few and to many workgroups, singly and two and four
    neighbours at a time; in the small ones a workgroup has so many of them that its groups take one each.  (The groups of a
    workgroup have one row each in the small matrices, two from 131 073 rows of four columns on, four from 262 145.)"""
    rng = np.random.default_rng(rows)
    lengths = rng.integers(0, 3, rows)
    for at in (0, rows // 2, rows - 20):
        block = slice(max(at, 0), min(at + 20, rows))
        lengths[block] = rng.choice([129, 130, 200, 512, 513, 600], block.stop - block.start)
    cols = 700
    p = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) if n > 2 else (7 * r + np.arange(n)) % (cols - 1)
                        for r, n in enumerate(lengths)] + [[]]).astype(np.int64)
    d = rng.standard_normal(i.size).astype(dtype)
    t = oracle.csr_transpose(rows, cols, d, i, p)
    for n in (4, 20, 70, 200) if rows < 100 else (4, 20, 70) if rows <= 40_000 else (4, 20):
        B, gC = randn(3, (cols, n), dtype), randn(4, (rows, n), dtype)
        C = host(ext.spdmm_forward(rows, cols, *to_dev(dev, d, i, p, B)))
        C_ref = oracle.spdmm_forward(rows, cols, d, i, p, B)
        kept = np.diff(p) <= 512
        assert_same(C[kept], C_ref[kept], f"n={n} C, rows in storage order")
        assert_close(C, C_ref, f"n={n} C")
        # the same rows as columns: both gradients
        ref = oracle.spdmm_backward(cols, rows, *t[:3], gC, B)
        got = ext.spdmm_backward(cols, rows, *to_dev(dev, *t[:3], gC, B))
        for g, w, what in zip(got, ref, ("grad_A", "grad_B")):
            assert_close(host(g), w, f"n={n} {what}")
        if mode == "eager":
            assert_same(host(got[1])[kept], ref[1][kept], f"n={n} grad_B, columns in storage order")
