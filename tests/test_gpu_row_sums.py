"""Rows summed from LDS several products at a time: at the lengths where a group of products ends, alone in their tile
and between short rows, the sum is that of the products taken one after the other."""
import numpy as np
import pytest

from numml_amd import _binding
from util import assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("around", [0, 3])
@pytest.mark.parametrize("long", [1, 15, 16, 17, 31, 32, 33, 47, 1000, 2047])
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
    assert_same(y, want, "y")
