"""The banded LU where the work changes hands: a value in the middle of a band that is not finite, a pivot that is zero or a
-0.0 ends the panel-wise elimination, and the column-wise one goes on behind the last panel that was written.

Rows and columns are those around a panel's edges (panels of eight), the first and last panel included; the reaches leave one
register of rows, two, the wider and the narrower rings, and no rows or columns beyond the next panel.  The factors are
compared bit for bit with the CPU oracle, signs of zeros included (cpp/sparse_csr_cpu.cpp:880-1016).
"""
import numpy as np
import pytest

import numml_amd
import oracle
from test_gpu_splu import NAMES, _banded
from util import assert_same, host, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n, below, above", [(41, 1, 1), (90, 8, 9), (150, 20, 24), (210, 56, 57), (210, 64, 64), (250, 92, 76), (120, 3, 70)])
def test_elimination_goes_on_column_by_column(dev, dtype, n, below, above):
    ext = numml_amd.load_compiled()
    r_of = lambda p: np.repeat(np.arange(n), np.diff(p))
    for special in ("zero pivot", "infinity", "not a number", "negative zero"):
        for row, col in ((7, 7), (8, 8), (17, 16), (24, 25), (39, 40), (n // 8 * 8 - 1, n // 8 * 8), (n - 1, n - 1)):
            if special == "zero pivot":
                col = row
            d, i, p = _banded(n, below, above, dtype, n + below, 0.5)
            r = r_of(p)
            if special == "zero pivot":
                # no product reaches this pivot: its row has nothing left of it
                d[(r == row) & (i <= row)] = 0.0
            else:
                d[(r == row) & (i == col)] = {"infinity": np.inf, "not a number": np.nan, "negative zero": -0.0}[special]
            print("case", n, below, above, np.dtype(dtype).name, special, row, col, flush=True)
            got, want = ext.splu(n, n, *to_dev(dev, d, i, p)), oracle.splu(n, n, d, i, p)
            for g, ref, what in zip(got, want, NAMES):
                g = host(g)
                assert_same(g, ref, f"{special} {row} {col} {what}")
                if g.dtype == dtype:
                    ok = ~np.isnan(ref)
                    assert np.array_equal(np.signbit(g[ok]), np.signbit(ref[ok])), f"{special} {row} {col} {what}: signs of zeros"
