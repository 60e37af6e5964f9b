"""Products whose rows leave the narrow hash tables: lengths on both sides of every table's limit,
columns in which many products meet, rows of B from empty to thousands of entries, columns packed
together and far apart.  Sums keep the order of A's row, so everything is compared bit for bit
against the serial loop, except rows longer than any table (added with atomics) and the gradient
of B (atomics): a sum of m products in any order is off by at most m * eps * sum |products|, and the
parity bound of the suite is above that for the lengths here."""
import numpy as np
import pytest
import torch

import numml_amd
import oracle
from numml_amd import generators as G
from numml_amd import numml_torch_cpp as ext
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu
DTYPES = [np.float32, np.float64]


def _csr(rows, cols, seed, dtype):
    indptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    indices = np.concatenate([np.asarray(r, np.int64) for r in rows] + [np.zeros(0, np.int64)])
    return randn(seed, indices.size, dtype), indices, indptr, (len(rows), cols)


def _lengths(lengths, spread, hub, dtype):
    """Row i of C has lengths[i] entries: B's row k holds column (k + 1) * spread and, with `hub`,
    column 0 in every third row, so that many products of a row meet there."""
    K = max(lengths)
    B = [([0] if hub and k % 3 == 0 else []) + [(k + 1) * spread] for k in range(K)]
    rng = np.random.default_rng(len(lengths) + spread)
    A = [np.sort(rng.choice(K, n - 1, replace=False)) if hub else np.arange(n) for n in lengths]
    return _csr(A, K, 1, dtype), _csr(B, (K + 1) * spread, 2, dtype)


def _blocks(dtype):
    """B's rows are runs of 0, 1, 300 and 5000 columns that overlap; columns packed in one corner
    with a single one far away."""
    cols = 3_000_000
    B = []
    for k in range(400):
        n = (0, 1, 300, 7)[k % 4] if k != 203 else 5000
        B.append(np.arange(k * 11, k * 11 + n))
    B[5] = np.concatenate([B[5], [cols - 1]])
    rng = np.random.default_rng(3)
    A = [np.arange(400), np.arange(0, 400, 2), np.arange(2, 400, 4), np.arange(0, 400, 4), np.arange(5, 60),
         np.sort(rng.choice(400, 130, replace=False)), [203], []]
    return _csr(A, 400, 4, dtype), _csr(B, cols, 5, dtype)


def _check(dev, a, b, dtype, exact=True):
    (ad, ai, ap, (ar, ac)), (bd, bi, bp, (br, bc)) = a, b
    Cd_ref, Ci_ref, Cp_ref = oracle.spgemm_forward(ar, ac, ad, ai, ap, br, bc, bd, bi, bp)
    gC = randn(9, Cd_ref.shape[0], dtype)
    gA_ref, gB_ref = oracle.spgemm_backward(gC, Ci_ref, Cp_ref, ar, ac, ad, ai, ap, br, bc, bd, bi, bp)
    AD, AI, AP, BD, BI, BP, GC = to_dev(dev, ad, ai, ap, bd, bi, bp, gC)
    Cd, Ci, Cp = ext.spgemm_forward(ar, ac, AD, AI, AP, br, bc, BD, BI, BP)
    assert_same(host(Cp), Cp_ref, "C_indptr")
    assert_same(host(Ci), Ci_ref, "C_indices")
    (assert_same if exact else assert_close)(host(Cd), Cd_ref, "C_data")
    for mode in ("planned", "atomic"):
        old_mode, ext.BACKWARD_MODE = ext.BACKWARD_MODE, mode
        try:
            gA, gB = ext.spgemm_backward(GC, Ci, Cp, ar, ac, AD, AI, AP, br, bc, BD, BI, BP)
        finally:
            ext.BACKWARD_MODE = old_mode
        assert_same(host(gA), gA_ref, f"grad_A ({mode})")
        assert_close(host(gB), gB_ref, f"grad_B ({mode})")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("spread", [1, 37])
def test_rows_at_the_limits_of_the_tables(dev, dtype, hub, spread):
    lengths = [n + d for n in (64, 128, 256, 512, 1024, 2048, 4096) for d in (0, 1)]
    _check(dev, *_lengths(lengths + lengths[::-1], spread, hub, dtype), dtype)


@pytest.mark.parametrize("dtype,most", [(np.float32, 16384), (np.float64, 10880)])
def test_rows_at_the_limit_of_a_compute_unit(dev, dtype, most):
    _check(dev, *_lengths([most, most - 1, 8192], 3, False, dtype), dtype)
    _check(dev, *_lengths([most + 1, 5000], 3, False, dtype), dtype, exact=False)


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_of_runs_and_of_packed_columns(dev, dtype):
    _check(dev, *_blocks(dtype), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_two_hop_graph(dev, dtype):
    a = G.powerlaw(6000, 6000, 60000, max_deg=1500, seed=7, dtype=dtype)
    _check(dev, a, a, dtype)


def _packed(lengths, cols, dtype):
    """Rows of C of about the given lengths: a run of columns somewhere, and the last column of all."""
    B = [np.arange(8 * k, 8 * k + 8) for k in range(4096)] + [[cols - 1]]
    rng = np.random.default_rng(6)
    A = [np.append(np.arange(s, s + (n - 1) // 8), 4096) for n in lengths for s in [int(rng.integers(0, 4096 - n // 8))]]
    return _csr(A, 4097, 6, dtype), _csr(B, cols, 7, dtype)


# a row in every shape of workgroup, nearly all of its columns in one bucket
@pytest.mark.parametrize("dtype,most", [(np.float32, 16384), (np.float64, 10880)])
@pytest.mark.parametrize("cols", [40_000, 20_000_000])
def test_a_column_far_from_the_others(dev, dtype, most, cols):
    _check(dev, *_packed([137, 200, 250, 264, 500, 520, 1000, 1024, 1032, 2000, 2050, 4000, 4100, 8200, most - 8, most],
                         cols, dtype), dtype)


def _time(dev, a, b):
    (ad, ai, ap, (ar, ac)), (bd, bi, bp, (br, bc)) = a, b
    AD, AI, AP, BD, BI, BP = to_dev(dev, ad, ai, ap, bd, bi, bp)
    best = float("inf")
    for _ in range(6):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        t0.record()
        ext.spgemm_forward(ar, ac, AD, AI, AP, br, bc, BD, BI, BP)
        t1.record()
        torch.cuda.synchronize()
        best = min(best, t0.elapsed_time(t1))
    return best


def test_the_time_of_packed_columns(dev):
    # a compare for every pair of columns took 13 times as long as columns that are spread out; sorting them 1.2
    rng = np.random.default_rng(8)
    spread = [np.sort(rng.choice(1_000_000, 8, replace=False)) for _ in range(4096)]
    A = [np.sort(rng.choice(4096, 500, replace=False)) for _ in range(300)]
    even = _time(dev, _csr(A, 4096, 1, np.float32), _csr(spread, 1_000_000, 2, np.float32))
    packed = _time(dev, *_packed([4000] * 300, 20_000_000, np.float32))
    assert packed < 4 * even, (packed, even)


def _hub(dtype, hub):
    """Two products per entry of A; with `hub` one of them in column 0, else all in columns of their own."""
    rng = np.random.default_rng(9)
    A = [np.sort(rng.choice(20_000, 4000, replace=False)) for _ in range(300)]
    B = [[0 if hub else 2 * k + 1, 2 * k + 2] for k in range(20_000)]
    return _csr(A, 20_000, 1, dtype), _csr(B, 40_001, 2, dtype)


def test_the_time_of_a_full_column(dev):
    # a turn of 1024 threads for every product in the full column took 8 times as long as products that do not meet, now 1.6
    even, full = _time(dev, *_hub(np.float64, False)), _time(dev, *_hub(np.float64, True))
    assert full < 4 * even, (full, even)


# products that meet in a few columns: 2 to 1000 of one chunk in a slot, several such slots among others, next to
# columns that nothing else adds to, in every shape of workgroup
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hubs", [1, 3, 40, 300])
def test_products_that_meet(dev, dtype, hubs):
    rng = np.random.default_rng(hubs)
    K = 3000
    B = [np.unique(np.append(rng.integers(0, hubs, rng.integers(1, 4)), [hubs + k, hubs + K + k])) for k in range(K)]
    A = [np.sort(rng.choice(K, n, replace=False)) for n in (60, 70, 120, 200, 250, 400, 500, 900, 1000, 1900, 2047, K)]
    _check(dev, _csr(A, K, 1, dtype), _csr(B, hubs + 2 * K, 2, dtype), dtype)


# the backward's lists of long rows: workgroups that look at 1, 2, 4 or 8 rows side by side, lengths of C's rows at
# both sides of each list's limits, any order
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 37, 700, 1500, 3000, 5000, 9001])
def test_rows_of_all_lengths_in_a_matrix(dev, dtype, rows):
    rng = np.random.default_rng(rows)
    lengths = np.where(rng.random(rows) < 0.9, rng.integers(0, 12, rows), 0)
    special = [64, 65, 512, 513, 2048, 2049, 2500]
    at = rng.permutation(rows)[:min(rows, 60)]
    lengths[at] = [special[k % 7] for k in range(at.size)]
    A = [np.sort(rng.choice(2600, n, replace=False)) for n in lengths]
    B = [[k] if k % 5 else [k, 2600 + k] for k in range(2600)]
    _check(dev, _csr(A, 2600, 1, dtype), _csr(B, 5200, 2, dtype), dtype)


def test_long_rows_behind_a_million_short_ones(dev):
    rows, K = 1_300_001, 3000
    lengths = np.ones(rows, np.int64)
    long = [3, 1_048_575, 1_048_576, 1_048_577, 1_100_000, 1_299_999, 1_300_000]
    lengths[long] = [100, 600, 3000, 2049, 513, 65, 2048]
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    indices = np.zeros(indptr[-1], np.int64)
    indices[indptr[:-1]] = np.arange(rows) % K
    for r in long:
        indices[indptr[r]:indptr[r + 1]] = np.arange(lengths[r])
    a = randn(1, indices.size, np.float64), indices, indptr, (rows, K)
    _check(dev, a, _csr([[k] for k in range(K)], K, 2, np.float64), np.float64)


def test_the_time_of_finding_no_long_rows(dev):
    # both gradients of a stencil's product take as long as the product; with a launch for each of four
    # shapes of long row that is not there they took 1.7 times as long
    c = numml_amd.load_compiled()
    d, i, p, (n, _) = G.poisson2d(300, np.float32)
    a = to_dev(dev, d, i, p)
    old = c.backward_mode()
    c.set_backward_mode("atomic")
    try:
        Cd, Ci, Cp = c.spgemm_forward(n, n, *a, n, n, *a)
        times = []
        for f in (lambda: c.spgemm_forward(n, n, *a, n, n, *a),
                  lambda: c.spgemm_backward(Cd, Ci, Cp, n, n, *a, n, n, *a)):
            best = float("inf")
            for _ in range(8):
                t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                torch.cuda.synchronize()
                t0.record()
                for _ in range(20):
                    f()
                t1.record()
                torch.cuda.synchronize()
                best = min(best, t0.elapsed_time(t1))
            times.append(best)
    finally:
        c.set_backward_mode(old)
    assert times[1] < 1.4 * times[0], times


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width, exact", [(300, True), (9000, True), (30_000, False)])
def test_more_products_than_any_table_holds(dev, dtype, width, exact):
    # 25 000 to 40 000 products a row, more such rows than there are workgroups with markers for them, beside rows
    # of every other length; what comes out fits a small table, a large one, or none
    rng = np.random.default_rng(width)
    B = [np.unique(rng.integers(0, width, 100)) for _ in range(2000)]
    A = [np.sort(rng.choice(2000, n, replace=False)) for n in [400, 1, 20, 300, 2, 90] * 24]
    _check(dev, _csr(A, 2000, 1, dtype), _csr(B, width, 2, dtype), dtype, exact)
