"""The banded LU where the work changes hands: a value in the middle of a band that is not finite or a pivot that is zero
ends the panel-wise elimination, and the column-wise one goes on behind the last panel that was written.  A -0.0 does
not end it: it keeps its sign until a product of two stored entries reaches it.

Rows and columns are those around a panel's edges (panels of eight), the first and last panel included; the reaches leave one
register of rows, two, the wider and the narrower rings, and no rows or columns beyond the next panel.  The factors are
compared bit for bit with the CPU oracle, signs of zeros included (cpp/sparse_csr_cpu.cpp:880-1016).
"""
import numpy as np
import pytest
import torch

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


def _masked(n, below, above, dtype, seed, holes, share):
    """A banded matrix of which `share` of the entries off the diagonal is masked by a product with zero: +0.0 and -0.0."""
    d, i, p = _banded(n, below, above, dtype, seed, holes)
    r = np.repeat(np.arange(n), np.diff(p))
    rng = np.random.default_rng(seed)
    # (rows and columns that are masked throughout among them: nothing ever reaches these entries)
    off = (r != i) & ((rng.random(d.size) < share) | (rng.random(n)[r] < share / 4) | (rng.random(n)[i] < share / 4))
    d[off] *= 0.
    d[np.flatnonzero(r != i)[[0, -1]]] = -0.
    return d, i, p


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n, below, above", [(9, 1, 1), (41, 1, 1), (90, 8, 9), (150, 20, 24), (210, 56, 57), (210, 64, 64), (250, 92, 76), (120, 3, 70),
                                             (120, 70, 3)])
def test_masked_matrices_keep_their_signs_of_zeros(dev, dtype, n, below, above):
    ext = numml_amd.load_compiled()
    for holes in (0.0, 0.6):
        for share in (0.05, 0.5, 0.95):
            d, i, p = _masked(n, below, above, dtype, n + below, holes, share)
            if share == 0.5:   # products that vanish: a -0 that is one of two stored entries counts
                d[d != 0] = np.where(np.abs(d[d != 0]) < 1, d[d != 0] * np.finfo(dtype).tiny, d[d != 0])
            got, want = ext.splu(n, n, *to_dev(dev, d, i, p)), oracle.splu(n, n, d, i, p)
            for g, ref, what in zip(got, want, NAMES):
                g = host(g)
                assert_same(g, ref, f"{holes} {share} {what}")
                if g.dtype == dtype:
                    assert np.array_equal(np.signbit(g), np.signbit(ref)), f"{holes} {share} {what}: signs of zeros"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("reach", [8, 60])
def test_a_negative_zero_costs_little(dev, dtype, reach):
    # It used to send the columns from it on to the column-wise kernel: four times the time of the whole factorisation.
    ext = numml_amd.load_compiled()
    n = 1200
    d, i, p = _banded(n, reach, reach, dtype, 3, 0.5)
    times = []
    for value in (0.0, -0.0):
        d[p[1]] = value                      # row 1, column 0 or the diagonal's neighbour
        args = to_dev(dev, d, i, p)
        for _ in range(2):
            ext.splu(n, n, *args)
        best = np.inf
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ext.splu(n, n, *args)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    assert times[1] < 1.8 * times[0], times
