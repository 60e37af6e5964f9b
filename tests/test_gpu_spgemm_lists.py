"""Products beyond the records, on a plan that lists their products (nm_spgemm_lists.hip): the serial loops' bits
for C and both gradients, at lengths around a tile of products (2048) and a workgroup's segments (256 and 2048),
and the limit beyond which the plan is refused."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from numml_amd import _binding, _lib
from numml_amd import generators as G
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(_binding.name != "compiled", reason="the plan policy lives in the compiled binding")]


def _csr(lengths, cols, seed, dtype):
    rng = np.random.default_rng(seed)
    p = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    i = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lengths] + [[]]).astype(np.int64)
    return rng.standard_normal(i.size).astype(dtype), i, p, (len(lengths), cols)


def _pairs(dtype):
    rng = np.random.default_rng(0)
    # rows of B of 0 to 300 entries among them more than the records take
    yield "mixed", _csr(rng.integers(0, 9, 700), 400, 1, dtype), _csr(rng.integers(0, 40, 400), 900, 2, dtype)
    yield "long rows of C", _csr([300, 0, 1, 40, 40, 0, 0], 400, 3, dtype), _csr(rng.integers(0, 60, 400), 5000, 4, dtype)
    # one row of A whose products fill a tile exactly, fall one short of it, and exceed it by one
    for extra in (-1, 0, 1):
        lengths = np.full(64, 32)
        lengths[7] += extra
        yield f"a tile {extra:+d}", _csr([64, 1], 64, 5, dtype), _csr(lengths, 4000, 6, dtype)
    # products that meet: few columns
    yield "few columns", _csr(rng.integers(0, 30, 300), 200, 7, dtype), _csr(rng.integers(1, 40, 200), 45, 8, dtype)
    # entries of C with one product each, just below and above a workgroup's 2048 segments
    for n in (2047, 2048, 2049):
        yield f"{n} entries of C", _csr([1, 0], 1, 9, dtype), _csr([n], 5000, 10, dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_the_serial_loops_bits(dev, dtype):
    ops = _binding.ops
    old = ops.backward_mode()
    ops.set_backward_mode("eager")
    try:
        for name, (ad, ai, ap, (ar, ac)), (bd, bi, bp, (br, bc)) in _pairs(dtype):
            ops.clear_plan_cache()
            ref = oracle.spgemm_forward(ar, ac, ad, ai, ap, br, bc, bd, bi, bp)
            gC = randn(11, ref[0].shape, dtype)
            gA_ref, gB_ref = oracle.spgemm_backward(gC, ref[1], ref[2], ar, ac, ad, ai, ap, br, bc, bd, bi, bp)
            A, B, Gd = to_dev(dev, ad, ai, ap), to_dev(dev, bd, bi, bp), to_dev(dev, gC)[0]
            for _ in range(2):      # (the first call makes the plan)
                C = ops.spgemm_forward(ar, ac, *A, br, bc, *B)
                for got, want, what in zip(C, ref, ("values", "columns", "row pointers")):
                    assert_same(host(got), want, f"{name}: {what}")
            both = ops.spgemm_backward(Gd, C[1], C[2], ar, ac, *A, br, bc, *B)
            assert ops.last_backward_paths()[1] == "product plan", name
            assert_same(host(both[0]), gA_ref, f"{name}: grad_A")
            assert_same(host(both[1]), gB_ref, f"{name}: grad_B")
            alone = ops.spgemm_backward(Gd, C[1], C[2], ar, ac, A[0].clone().requires_grad_(True), *A[1:], br, bc, *B)
            assert alone[1] is None and torch.equal(alone[0], both[0])
    finally:
        ops.set_backward_mode(old)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_a_busy_workgroup_is_refused(dev, dtype):
    """A hub column of A that meets a long row of B: no plan, the stateless kernels as before."""
    ops = _binding.ops
    ops.clear_plan_cache()
    rows = 700
    a = [np.array([0]) if r % 2 else np.array([0, 1 + r]) for r in range(rows)]
    ap = np.concatenate([[0], np.cumsum([r.size for r in a])]).astype(np.int64)
    ai = np.concatenate(a).astype(np.int64)
    ad = randn(1, ai.size, dtype)
    lengths = np.full(rows + 1, 2)
    lengths[0] = 300
    bd, bi, bp, (br, bc) = _csr(lengths, 4000, 2, dtype)
    A, B = to_dev(dev, ad, ai, ap), to_dev(dev, bd, bi, bp)
    ref = oracle.spgemm_forward(rows, br, ad, ai, ap, br, bc, bd, bi, bp)
    gC = randn(3, ref[0].shape, dtype)
    want = oracle.spgemm_backward(gC, ref[1], ref[2], rows, br, ad, ai, ap, br, bc, bd, bi, bp)
    for _ in range(3):
        C = ops.spgemm_forward(rows, br, *A, br, bc, *B)
        assert_same(host(C[0]), ref[0], "values")
        got = ops.spgemm_backward(to_dev(dev, gC)[0], C[1], C[2], rows, br, *A, br, bc, *B)
        assert ops.last_backward_paths()[1] != "product plan"
        for g, w in zip(got, want):
            assert_close(host(g), w, "gradient")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [127, 128, 129, 4096, 4097, 9000, 40_000])
def test_an_entry_of_many_products(dev, dtype, n):
    """One entry of C with n products, in the serial loop's order (put there by rank below 128 of them, sorted in LDS
    up to 4096 and in pieces beyond).  The row of 40 entries keeps the product off the records."""
    ops = _binding.ops
    ops.clear_plan_cache()
    ai, ap = np.arange(n), np.array([0, n], np.int64)
    lengths = np.ones(n, np.int64)
    lengths[n // 3] = 40
    bp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    bi = np.concatenate([np.arange(m) for m in lengths]).astype(np.int64)
    ad, bd = randn(n, n, dtype), randn(n + 1, bi.size, dtype)
    ref = oracle.spgemm_forward(1, n, ad, ai, ap, n, 40, bd, bi, bp)
    gC = randn(n + 2, ref[0].shape, dtype)
    want = oracle.spgemm_backward(gC, ref[1], ref[2], 1, n, ad, ai, ap, n, 40, bd, bi, bp)
    A, B, Gd = to_dev(dev, ad, ai, ap), to_dev(dev, bd, bi, bp), to_dev(dev, gC)[0]
    for k in range(3):
        C = ops.spgemm_forward(1, n, *A, n, 40, *B)
        (assert_same if k == 2 else assert_close)(host(C[0]), ref[0], "values")
    got = ops.spgemm_backward(Gd, C[1], C[2], 1, n, *A, n, 40, *B)
    assert ops.last_backward_paths()[1] == "product plan"
    for g, w in zip(got, want):
        assert_same(host(g), w, "gradient")


def _build(dev, A, B, C, products):
    """`usable` of nm_spgemm_lists_build for patterns (indices, indptr, shape)."""
    L, plan, work, usable = _lib.lib(), ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_int(-1)
    (ai, ap, (m, k)), (bi, bp, _), (ci, cp, _) = A, B, C
    t = [to_dev(dev, *x[:2]) for x in (A, B, C)]
    assert L.nm_csr_transpose_plan_bytes(m, k, ai.size, plan, work) == 0
    tp, tw = (torch.empty(s.value, dtype=torch.uint8, device=dev) for s in (plan, work))
    assert L.nm_csr_transpose_plan_build(m, k, ai.size, t[0][0].data_ptr(), t[0][1].data_ptr(), tp.data_ptr(), plan, tw.data_ptr(), work, None) == 0
    assert L.nm_spgemm_lists_bytes(k, ai.size, bi.size, ci.size, products, plan, work) == 0
    lp, lw = (torch.empty(s.value, dtype=torch.uint8, device=dev) for s in (plan, work))
    ptrs = [x.data_ptr() for pair in t for x in pair]
    assert L.nm_spgemm_lists_build(m, k, ai.size, bi.size, ci.size, products, *ptrs, tp.data_ptr(), lp.data_ptr(), plan,
                                   lw.data_ptr(), work, usable, None) == 0
    torch.cuda.synchronize()
    return usable.value


def test_what_is_refused_depends_on_the_counts(dev):
    """On either side of 65 536 products in a workgroup of C (one entry, and many entries that share one) and of 16 384 and
    65 536 in one of a gradient."""
    rows = lambda lengths, cols, pick: (np.concatenate([pick(r, n) for r, n in enumerate(lengths)]).astype(np.int64),
                                        np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64), (len(lengths), cols))
    first = lambda r, n: np.arange(n)
    full = lambda m, n: rows([n] * m, n, first)
    # one entry of C with all products, alone (known from the sizes) and among 2048 more entries (counted)
    for n, usable in ((65_536, 1), (65_537, 0)):
        assert _build(dev, full(1, n), rows([1] * n, 1, first), full(1, 1), n) == usable
    more = 2048
    for n, usable in ((65_536 - 255, 1), (65_536 - 254, 0)):
        A = rows([n] + [1] * more, n + more, lambda r, m: np.arange(m) if r == 0 else np.array([n + r - 1]))
        B = rows([1] * (n + more), 1, first)
        assert _build(dev, A, B, full(1 + more, 1), n + more) == usable
    # 256 entries of A with n products each, as many entries of B (one row) with 256
    for n, usable in ((64, 1), (65, 2), (256, 2), (257, 0)):
        assert _build(dev, full(256, 1), full(1, n), full(256, n), 256 * n) == usable


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n, planned", [(64, True), (65, False)])
def test_gradients_of_busy_workgroups_go_without_the_plan(dev, dtype, n, planned):
    ops = _binding.ops
    ops.clear_plan_cache()
    ad, bd = randn(1, 256, dtype), randn(2, n, dtype)
    ai, ap = np.zeros(256, np.int64), np.arange(257)
    bi, bp = np.arange(n), np.array([0, n], np.int64)
    A, B = to_dev(dev, ad, ai, ap), to_dev(dev, bd, bi, bp)
    ref = oracle.spgemm_forward(256, 1, ad, ai, ap, 1, n, bd, bi, bp)
    gC = randn(3, ref[0].shape, dtype)
    want = oracle.spgemm_backward(gC, ref[1], ref[2], 256, 1, ad, ai, ap, 1, n, bd, bi, bp)
    for k in range(3):
        C = ops.spgemm_forward(256, 1, *A, 1, n, *B)
        assert_same(host(C[0]), ref[0], "values")
        got = ops.spgemm_backward(to_dev(dev, gC)[0], C[1], C[2], 256, 1, *A, 1, n, *B)
        for g, w in zip(got, want):
            assert_close(host(g), w, "gradient")
    assert (ops.last_backward_paths()[1] == "product plan") == planned
    built = ops.plan_cache_stats()[0]
    C2 = ops.spgemm_forward(256, 1, *A, 1, n, *B)
    assert C2[1].data_ptr() == C[1].data_ptr() and ops.plan_cache_stats()[0] == built, "the forward is on the plan"


def test_sizes_and_memory_are_checked(dev):
    L = _lib.lib()
    n = ctypes.c_int64()
    plan, work = ctypes.c_size_t(), ctypes.c_size_t()
    assert L.nm_spgemm_lists_bytes(10, 5, 5, 5, 2 ** 31, plan, work) != 0
    assert L.nm_spgemm_lists_bytes(10, 5, 5, 5, 25, plan, work) == 0 and plan.value > 0 and work.value > 0
    I, P = to_dev(dev, np.array([0, 1, 1], np.int64), np.array([0, 3, 5], np.int64))
    room = torch.empty(4096, dtype=torch.uint8, device=dev)
    assert L.nm_spgemm_lists_products(3, I.data_ptr(), P.data_ptr(), room.data_ptr(), 16, n, None) != 0
    assert L.nm_spgemm_lists_products(3, I.data_ptr(), P.data_ptr(), room.data_ptr(), 4096, n, None) == 0 and n.value == 7
