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
