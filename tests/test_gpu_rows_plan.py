"""Matrix-vector products without gradients on the part of the plan that they read: from the third product with the
same tensors on, the bits of the products before, and where it is not made or no longer taken."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from numml_amd import _binding, _lib
from numml_amd import generators as G
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu
needs_policy = pytest.mark.skipif(_binding.name != "compiled", reason="the plan policy lives in the compiled binding")


@pytest.fixture(autouse=True)
def default_mode():
    old = _binding.backward_mode()
    _binding.set_backward_mode("planned")
    yield
    _binding.set_backward_mode(old)


def _some_long(rows, dtype):
    """Three random columns a row, up to 6000 in seven of them."""
    rng = np.random.default_rng(rows)
    lens = np.full(rows, 3)
    lens[[0, 15, 16, 5000, rows // 2, rows - 600, rows - 1]] = [31, 32, 2000, 4096, 4097, 6000, 5]
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    i = rng.integers(0, rows, p[-1])
    return randn(5, p[-1], dtype), i, p, (rows, rows)


def _band_with_long_rows(dtype):
    """Rows of four entries, of 31 to 200 here and there, all within 300 columns: every block has a staging list."""
    rng = np.random.default_rng(9)
    lens = np.full(3072, 4)
    lens[[0, 1, 2, 3, 64, 700, 701, 1400, 2047, 2048, 3071]] = [31, 32, 33, 64, 65, 200, 129, 63, 128, 32, 40]
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    i = np.concatenate([np.sort(max(0, min(r - 150, 2772)) + rng.choice(300, n, replace=False)) for r, n in enumerate(lens)])
    return randn(5, p[-1], dtype), i.astype(np.int64), p, (3072, 3072)


def _mixed(rows, width, dtype):
    """Rows of 1 to 40 entries, 20 on average, somewhere in `width` columns that move along the diagonal."""
    rng = np.random.default_rng(width)
    lens = rng.integers(1, 41, rows)
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    i = np.repeat(np.arange(rows) * (rows - width) // rows, lens) + rng.integers(0, width, p[-1])
    return randn(6, p[-1], dtype), i.astype(np.int64), p, (rows, rows)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", ["band with long rows", "grid", "wide band", "scattered", "ragged", "one row", "511 rows", "513 rows", "65536 rows",
                                  "65535 rows, some long", "70000 rows, some long", "65535 rows of 1 to 40", "65536 rows of 1 to 40",
                                  "65536 rows of 1 to 40, all columns"])
def test_the_bits_of_the_plain_kernel(dev, dtype, case):
    d, i, p, (rows, cols) = {
        "band with long rows": lambda: _band_with_long_rows(dtype),
        "grid": lambda: G.poisson2d(40, dtype, jitter_seed=1),
        "wide band": lambda: G.laplace3d(20, dtype, jitter_seed=1),
        "scattered": lambda: G.random_csr(3000, 90_000, 0.0003, 2, dtype),
        "ragged": lambda: G.ragged_csr(2000, 1500, 31, 8, dtype, min_len=0),
        "one row": lambda: G.random_csr(1, 50, 0.5, 3, dtype, empty_rows=False),
        "511 rows": lambda: G.tridiag(511, dtype),
        "513 rows": lambda: G.tridiag(513, dtype),
        "65536 rows": lambda: G.poisson2d(256, dtype, jitter_seed=1),
        "65535 rows, some long": lambda: _some_long(65535, dtype),
        "70000 rows, some long": lambda: _some_long(70000, dtype),
        "65535 rows of 1 to 40": lambda: _mixed(65535, 500, dtype),
        "65536 rows of 1 to 40": lambda: _mixed(65536, 500, dtype),
        "65536 rows of 1 to 40, all columns": lambda: _mixed(65536, 65536, dtype),
    }[case]()
    nnz = d.size
    x = randn(4, cols, dtype)
    D, I, P, X = to_dev(dev, d, i, p, x)
    L, size, info = _lib.lib(), ctypes.c_size_t(), (ctypes.c_int32 * 16)()
    assert L.nm_spgemv_rows_plan_bytes(rows, cols, nnz, size) == 0
    plan = torch.empty(size.value, dtype=torch.uint8, device=dev)
    args = (rows, cols, nnz, I.data_ptr(), P.data_ptr(), plan.data_ptr())
    assert L.nm_spgemv_rows_plan_build(*args, size.value - 1, info, None) != 0
    assert L.nm_spgemv_rows_plan_build(*args, size, info, None) == 0
    assert info[7] == np.diff(p).max()
    if case == "band with long rows":
        assert info[4] == 6
    kind = 0 if dtype == np.float32 else 1
    plain = torch.empty(rows, dtype=D.dtype, device=dev)
    assert L.nm_spgemv_forward(kind, rows, cols, nnz, D.data_ptr(), I.data_ptr(), P.data_ptr(), X.data_ptr(), plain.data_ptr(), None) == 0
    want = host(plain)
    assert_close(want, oracle.spgemv_forward(rows, cols, d, i, p, x), case)
    for lists in (0, 1):
        y = torch.full((rows,), 7, dtype=D.dtype, device=dev)
        assert L.nm_spgemv_forward_rows(kind, lists, rows, cols, nnz, D.data_ptr(), plan.data_ptr(), X.data_ptr(), y.data_ptr(), None) == 0
        assert_same(host(y), want, f"{case}, lists={lists}")


@needs_policy
def test_from_the_third_product_on(dev):
    ops = _binding.ops
    d, i, p, (rows, cols) = G.poisson2d(480, np.float64, jitter_seed=1)      # 1.15 M entries
    D, I, P, X = to_dev(dev, d, i, p, randn(1, cols, np.float64))
    want = oracle.spgemv_forward(rows, cols, d, i, p, host(X))

    def products(n, *m):
        out = []
        for _ in range(n):
            assert_same(host(ops.spgemv_forward(rows, cols, *m, X)), want, "y")
            out.append(ops.plan_cache_size())
        return out
    ops.clear_plan_cache()
    assert products(5, D, I, P) == [0, 0, 1, 1, 1]
    # a clone is counted anew and finds the plan by content
    assert products(4, D, I.clone(), P.clone()) == [1] * 4
    # edited in place: seen as other tensors; the product is of the edited pattern
    J = I.clone()
    products(3, D, J, P)
    J[0], J[1] = int(J[1]), int(J[0])
    E = D.clone()
    E[0], E[1] = D[1], D[0]
    y = ops.spgemv_forward(rows, cols, E, J, P, X)
    assert np.allclose(host(y), want)
    # gradients make the whole plan, which the forward takes then
    for _ in range(3):
        ops.spgemv_backward(X, rows, cols, D, I, P, X)
        assert_same(host(ops.spgemv_forward(rows, cols, D, I, P, X)), want, "y")
    # never where plans are switched off, for small matrices, and in inference mode
    ops.clear_plan_cache()
    ops.set_backward_mode("atomic")
    assert products(4, D, I, P) == [0] * 4
    ops.set_backward_mode("planned")
    with torch.inference_mode():
        assert products(4, D.clone(), I.clone(), P.clone()) == [0] * 4
    s = to_dev(dev, *G.tridiag(100, np.float64)[:3])
    for _ in range(4):
        ops.spgemv_forward(100, 100, *s, X[:100])
    assert ops.plan_cache_size() == 0


@needs_policy
def test_under_capture_nothing_is_made(dev):
    ops = _binding.ops
    ops.clear_plan_cache()
    d, i, p, (rows, cols) = G.poisson2d(480, np.float32, jitter_seed=1)
    D, I, P, X = to_dev(dev, d, i, p, randn(1, cols, np.float32))
    for before in (2, 4):       # captured by the plain kernel, then on the plan
        y = None
        for _ in range(before):
            y = ops.spgemv_forward(rows, cols, D, I, P, X)
        torch.cuda.synchronize()
        held = ops.plan_cache_size()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            z = ops.spgemv_forward(rows, cols, D, I, P, X)
        assert ops.plan_cache_size() == held
        for k in range(3):
            X.copy_(torch.from_numpy(randn(10 + k, cols, np.float32)))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(z, ops.spgemv_forward(rows, cols, D, I, P, X))


@needs_policy
def test_a_plan_that_does_not_stay_is_not_made_on_every_product(dev):
    ops = _binding.ops
    d, i, p, (rows, cols) = G.poisson2d(480, np.float32, jitter_seed=1)
    D, I, P, X = to_dev(dev, d, i, p, randn(1, cols, np.float32))
    other = I.clone()
    other[0], other[1] = int(I[1]), int(I[0])       # another content: a plan of its own
    size = ctypes.c_size_t()
    assert _lib.lib().nm_spgemv_rows_plan_bytes(rows, cols, d.size, size) == 0

    def built(products, *index):
        before = ops.plan_cache_stats()[0]
        for _ in range(products):
            for j in index:
                ops.spgemv_forward(rows, cols, D, j, P, X)
        return ops.plan_cache_stats()[0] - before
    try:
        ops.clear_plan_cache()
        ops.set_plan_cache_limit(size.value * 3 // 2)           # room for one of the two
        assert built(20, I, other) == 2
        assert 1 <= built(200, I, other) <= 6                   # (every second of 400 without a bound)
        ops.clear_plan_cache()
        ops.set_plan_cache_limit(size.value - 1)
        assert built(20, I) == 0
        ops.set_plan_cache_limit(size.value + 64)               # (the plan's tensor may be a little larger than asked for)
        assert built(64, I) == 1 and built(64, I) == 0
    finally:
        ops.set_plan_cache_limit(4 << 30)
        ops.clear_plan_cache()


@needs_policy
def test_no_memory_for_the_plan(dev):
    """The product is made without it."""
    ops = _binding.ops
    d, i, p, (rows, cols) = G.poisson2d(1000, np.float32, jitter_seed=1)        # 5 M entries, a plan of 30 MB
    D, I, P, X = to_dev(dev, d, i, p, randn(1, cols, np.float32))
    ops.clear_plan_cache()
    want = [ops.spgemv_forward(rows, cols, D, I, P, X) for _ in range(2)][0]
    out = torch.empty_like(want)
    room = torch.empty(20 << 20, dtype=torch.uint8, device=dev)        # for the products
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    taken = []
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (2 << 20)) / torch.cuda.get_device_properties(0).total_memory)
        try:
            while len(taken) < 4096:        # what earlier work has left free inside its blocks
                taken.append(torch.empty(24 << 20, dtype=torch.uint8, device=dev))
        except torch.cuda.OutOfMemoryError:
            pass
        del room
        for _ in range(3):
            out.copy_(ops.spgemv_forward(rows, cols, D, I, P, X))
        assert ops.plan_cache_size() == 0
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, want)
