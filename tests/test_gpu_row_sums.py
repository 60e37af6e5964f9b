"""Rows summed from LDS several products at a time: at the lengths where a group of products ends, alone in their tile
and between short rows, the sum is that of the products taken one after the other; from 32 products on that of a
wavefront's 64 partial sums."""
import numpy as np
import pytest

from numml_amd import _binding
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("around", [0, 3])
@pytest.mark.parametrize("long", [1, 3, 4, 5, 15, 16, 17, 21, 31, 32, 33, 47, 63, 64, 65, 127, 1000, 2047])
def test_a_row_is_summed_in_order(dev, dtype, around, long):
    cols = 2500
    lens = np.array([around] * 100 + [long] + [around] * 99)
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rng = np.random.default_rng(long)
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lens]).astype(np.int64)
    d, x = randn(1, i.size, dtype), randn(2, cols, dtype)
    y = host(_binding.ops.spgemv_forward(lens.size, cols, *to_dev(dev, d, i, p, x)))
    prod = d * x[i]
    want = np.zeros(lens.size, dtype)
    for r in range(lens.size):
        for v in prod[p[r]:p[r + 1]]:
            want[r] += v
    short = lens < 32
    assert_same(y[short], want[short], "y")
    assert_close(y, want, "y")
    # the same bits wherever the row lies
    i2, lens2 = np.concatenate([i, i]), np.concatenate([lens, lens])
    p2 = np.concatenate([[0], np.cumsum(lens2)]).astype(np.int64)
    z = host(_binding.ops.spgemv_forward(lens2.size, cols, *to_dev(dev, np.concatenate([d, d]), i2, p2, x)))
    assert_same(z, np.concatenate([y, y]), "the row in another place")


def _in_parts(terms):
    """The order of long rows: term k to part k % 64, the parts pairwise."""
    parts = np.zeros(64, terms.dtype)
    for k, v in enumerate(terms):
        parts[k % 64] += v
    while parts.size > 1:
        parts = parts[0::2] + parts[1::2]
    return parts[0]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lengths", [[32], [33], [40], [63], [64], [65], [71, 72, 73], [127], [128], [129], [150], [32, 128], [5, 129, 64, 31],
                                     list(range(20, 140, 3))])
@pytest.mark.parametrize("rows", [1, 5, 6, 24, 150, 700])
def test_long_rows_have_one_order(dev, dtype, lengths, rows):
    """By the wavefront where it has few of them, by a lane each where it has many: the same bits, in every kernel that
    sums rows."""
    cols = 2500
    lens = np.resize(np.array(lengths), rows)
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rng = np.random.default_rng(rows)
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lens]).astype(np.int64)
    d, x = randn(1, i.size, dtype), randn(2, cols, dtype)
    ops, (D, I, P, X) = _binding.ops, to_dev(dev, d, i, p, x)

    def order(terms):
        return np.array([_in_parts(terms[b:e]) if e - b >= 32 else np.add.reduce(terms[b:e], initial=dtype(0)) if e - b < 2 else
                         np.add.accumulate(np.concatenate([[dtype(0)], terms[b:e]]))[-1] for b, e in zip(p[:-1], p[1:])], dtype)
    want = order(d * x[i])
    assert_same(host(ops.spgemv_forward(rows, cols, D, I, P, X)), want, "without a plan")
    assert_same(host(ops.csr_row_sum_forward(rows, cols, D, I, P)), order(d), "row sums")
    old = _binding.backward_mode()
    _binding.set_backward_mode("eager")
    try:
        # the transpose, whose columns are these rows
        t = _csr_transpose(d, i, p, cols)
        G = to_dev(dev, *t)
        gx = ops.spgemv_backward(X, cols, rows, *G, to_dev(dev, np.zeros(rows, dtype))[0])[1]
        assert_same(host(gx), order(x[i] * d), "gradient by columns")
        ops.spgemv_backward(to_dev(dev, np.zeros(rows, dtype))[0], rows, cols, D, I, P, X)
        assert_same(host(ops.spgemv_forward(rows, cols, D, I, P, X)), want, "on the plan")
    finally:
        _binding.set_backward_mode(old)


def _csr_transpose(d, i, p, cols):
    rows = np.repeat(np.arange(p.size - 1), np.diff(p))
    o = np.argsort(i, kind="stable")
    return d[o], rows[o].astype(np.int64), np.concatenate([[0], np.cumsum(np.bincount(i, minlength=cols))]).astype(np.int64)
