"""SpMV forward without a plan, whose lanes take two entries of the 64-bit structure at a time: blocks of rows whose entries
are none, one, an odd number, exactly what the tile holds and one more or less, that start at odd positions, and whose
arrays start at an odd element of their allocation.  Bit for bit the serial loop (cpp/sparse_csr_cpu.cpp:29-35)."""
import numpy as np
import pytest
import torch

import oracle
from numml_amd import numml_torch_cpp as ext
from util import assert_same, host, to_dev

pytestmark = pytest.mark.gpu


def _lengths(kind, rng):
    if kind == "one row, one entry":
        return [1]
    if kind == "no entries":
        return [0] * 700
    if kind == "odd blocks":                      # 512 rows of 5 and one of 6: the next block starts at an odd position
        return [5] * 511 + [4] + [5] * 511 + [6] + [3] * 513
    if kind == "around the tile":                 # 512 rows of 6 are 3072 entries
        return [6] * 512 + [6] * 511 + [5] + [6] * 511 + [7] + [6] * 100
    if kind == "empty blocks between":
        return [0] * 512 + [3] * 5 + [0] * 1019 + [1] + [0] * 511
    return list(rng.integers(0, 12, 1700))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["one row, one entry", "no entries", "odd blocks", "around the tile", "empty blocks between", "random"])
def test_two_entries_at_a_time(dev, dtype, kind):
    rng = np.random.default_rng(7)
    n = np.array(_lengths(kind, rng))
    rows, cols = n.size, 900
    p = np.concatenate(([0], np.cumsum(n))).astype(np.int64)
    i = rng.integers(0, cols, p[-1]).astype(np.int64)
    d, x = rng.uniform(-1, 1, p[-1]).astype(dtype), rng.uniform(-1, 1, cols).astype(dtype)
    print("case", kind, np.dtype(dtype).name, flush=True)
    want = oracle.spgemv_forward(rows, cols, d, i, p, x)
    D, I, P, X = to_dev(dev, d, i, p, x)
    assert_same(host(ext.spgemv_forward(rows, cols, D, I, P, X)), want, kind)
    shifted = lambda t: torch.cat([t[:1], t])[1:] if t.numel() else t
    assert_same(host(ext.spgemv_forward(rows, cols, shifted(D), shifted(I), P, X)), want, kind + ", shifted")
