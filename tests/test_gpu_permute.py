"""The backward of sparse times dense with the values brought into column-major order beforehand
(nm_spdmm_backward_staged): the bits of nm_spdmm_backward_planned, at sizes around a bin and a tile
(4096, 8192 and 16384 entries), and the default mode's choice of it."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from numml_amd import _binding, _lib
from numml_amd import numml_torch_cpp as ext
from util import assert_close, assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, nnz, dtype, dev):
    """nnz entries at random columns (a row may name a column twice)."""
    gen = torch.Generator(device="cuda").manual_seed(nnz)
    row = torch.sort(torch.randint(rows, (nnz,), generator=gen, device=dev))[0]
    P = torch.zeros(rows + 1, dtype=torch.int64, device=dev)
    P[1:] = torch.cumsum(torch.bincount(row, minlength=rows), 0)
    I = torch.sort(row * cols + torch.randint(cols, (nnz,), generator=gen, device=dev))[0] % cols
    D = torch.randn(nnz, generator=gen, device=dev, dtype=torch.float32 if dtype == np.float32 else torch.float64)
    return D, I, P


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nnz", [1, 63, 4095, 4096, 4097, 12000, (2 << 20), (2 << 20) + 1, (8 << 20) - 1, (8 << 20) + 5])
def test_same_bits_as_the_plan_alone(dev, dtype, nnz):
    L = _lib.lib()
    rows, cols = max(nnz // 7, 1), max(nnz // 5, 1)
    n = 5 if nnz < 100_000 else 2
    D, I, P = _matrix(rows, cols, nnz, dtype, dev)
    B = torch.randn(cols, n, device=dev, dtype=D.dtype)
    gC = torch.randn(rows, n, device=dev, dtype=D.dtype)
    plan = ext._transpose_plan(I, P, rows, cols, dev)
    pb, wb, sb = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    assert L.nm_permute_plan_bytes(nnz, pb, wb) == 0 and L.nm_spdmm_staged_bytes(ext._dt(D), nnz, sb) == 0
    perm, work, room = (torch.empty(max(b.value, 8), dtype=torch.uint8, device=dev) for b in (pb, wb, sb))
    assert L.nm_permute_plan_build(rows, cols, nnz, plan.mem.data_ptr(), perm.data_ptr(), pb, work.data_ptr(), wb, None) == 0
    out = {}
    for both in (True, False):
        for staged in (True, False):
            gA, gB = torch.full_like(D, 7), torch.full((cols, n), 7, device=dev, dtype=D.dtype)
            tail = (B.data_ptr(), n, gC.data_ptr(), n, n, gA.data_ptr() if both else None, gB.data_ptr(), n, None)
            if staged:
                rc = L.nm_spdmm_backward_staged(ext._dt(D), rows, cols, nnz, D.data_ptr(), plan.mem.data_ptr(),
                                                perm.data_ptr(), room.data_ptr(), sb, *tail)
            else:
                rc = L.nm_spdmm_backward_planned(ext._dt(D), rows, cols, nnz, D.data_ptr(), I.data_ptr(), P.data_ptr(),
                                                 plan.mem.data_ptr(), *tail)
            assert rc == 0, L.nm_last_error()
            out[staged] = (gA, gB)
        torch.cuda.synchronize()
        assert torch.equal(out[True][1], out[False][1]), "grad_B"
        assert torch.equal(out[True][0], out[False][0]), "grad_A"
    if nnz < 100_000:
        ref = oracle.spdmm_backward(rows, cols, host(D), host(I), host(P), host(B), host(gC))
        assert_same(host(out[True][1]), ref[1], "grad_B against the oracle")
    # memory that is too small, operands that are too wide and missing outputs are refused
    bad = (B.data_ptr(), n, gC.data_ptr(), n, n, None, gB.data_ptr(), n, None)
    args = (ext._dt(D), rows, cols, nnz, D.data_ptr(), plan.mem.data_ptr(), perm.data_ptr(), room.data_ptr())
    assert L.nm_spdmm_backward_staged(*args, sb.value - 1, *bad) != 0
    assert L.nm_spdmm_backward_staged(*args, sb, B.data_ptr(), 300, gC.data_ptr(), 300, 300, None, gB.data_ptr(), 300, None) != 0
    assert L.nm_spdmm_backward_staged(*args, sb, B.data_ptr(), n, gC.data_ptr(), n, n, gA.data_ptr(), None, n, None) != 0


def test_default_mode_takes_it_at_the_third_backward(dev):
    """...of a pattern whose columns are scattered, and never for a banded one of the same size."""
    ops = _binding.ops
    if _binding.name == "ctypes":
        pytest.skip("the policy lives in the compiled binding")
    old = ops.backward_mode()
    ops.set_backward_mode("planned")
    try:
        for scattered in (True, False):
            ops.clear_plan_cache()
            rows = 200_000
            D, I, P = _matrix(rows, rows, 1_500_000, np.float32, dev)
            if not scattered:
                row = torch.repeat_interleave(torch.arange(rows, device=dev), P[1:] - P[:-1])
                I = torch.sort(row * rows + (row + I % 50).clamp_max(rows - 1))[0] % rows
            B, gC = to_dev(dev, randn(1, (rows, 4), np.float32), randn(2, (rows, 4), np.float32))
            got, built = [], []
            for _ in range(4):
                got.append(ops.spdmm_backward(rows, rows, D, I, P, B, gC))
                built.append(ops.plan_cache_stats()[0])
            steps = [b - a for a, b in zip(built, built[1:])]
            assert steps == ([1, 1, 0] if scattered else [1, 0, 0])
            for a, b in got[2:]:
                assert torch.equal(a, got[1][0]) and torch.equal(b, got[1][1])
            assert_close(host(got[0][0]), host(got[3][0]), "grad_A against the stateless kernels")
            assert_close(host(got[0][1]), host(got[3][1]), "grad_B against the stateless kernels")
    finally:
        ops.set_backward_mode(old)
        ops.clear_plan_cache()


@pytest.mark.skipif(_binding.name != "compiled", reason="the plan policy lives in the compiled binding")
@pytest.mark.parametrize("dtype,both,rows,cols,nnz,want", [
    (np.float32, True, 8191, 200_000, 1_200_000, False), (np.float32, True, 8192, 200_000, 1_200_000, True),
    (np.float64, True, 4000, 120_001, 1_200_000, False), (np.float64, True, 4000, 120_000, 1_200_000, True),
    (np.float32, True, 127, 30_000, 1_200_000, False), (np.float32, True, 128, 30_000, 1_200_000, True),
    (np.float32, False, 4095, 500_000, 3_200_000, False), (np.float32, False, 4096, 500_000, 3_200_000, True),
    (np.float64, False, 32767, 500_000, 3_200_000, False), (np.float64, False, 32768, 500_000, 3_200_000, True),
    (np.float64, False, 1023, 32_000, 3_200_000, False), (np.float64, False, 1024, 32_000, 3_200_000, True)])
def test_vectors_go_through_the_order_where_there_are_rows_enough(dev, dtype, both, rows, cols, nnz, want):
    ops = _binding.ops
    D, I, P = _matrix(rows, cols, nnz, dtype, dev)
    x, g = torch.randn(cols, device=dev, dtype=D.dtype), torch.randn(rows, device=dev, dtype=D.dtype)
    old = ops.backward_mode()
    ops.set_backward_mode("planned")
    ops.clear_plan_cache()
    X = x if both else x.clone().requires_grad_(True)
    size, got = [], []
    for _ in range(4):
        got = ops.spgemv_backward(g, rows, cols, D, I, P, X)
        size.append(ops.plan_cache_size())
    ops.set_backward_mode(old)
    ops.clear_plan_cache()
    assert size == [0, 1, 2, 2] if want else size == [0, 1, 1, 1], size
    row = torch.repeat_interleave(torch.arange(rows, device=dev), P[1:] - P[:-1])
    terms = g[row].double() * D.double()
    ref = torch.zeros(cols, dtype=torch.float64, device=dev).index_add_(0, I, terms)
    size_of = torch.zeros(cols, dtype=torch.float64, device=dev).index_add_(0, I, terms.abs())
    count = torch.bincount(I, minlength=cols)
    # sums of n terms in any order: 2 n eps times the sum of their sizes
    assert ((got[1].double() - ref).abs() <= 2 * torch.finfo(D.dtype).eps * (count + 1) * size_of).all()
    if both:
        assert torch.equal(got[0], g[row] * x[I])


@pytest.mark.skipif(_binding.name != "compiled", reason="the plan policy lives in the compiled binding")
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,nnz,want", [(16_383, 1 << 20, False), (16_384, 1 << 20, True), (16_384, (1 << 20) - 1, False)])
def test_dense_operands_go_through_the_order_where_there_are_rows_and_entries_enough(dev, dtype, rows, nnz, want):
    ops, cols, n = _binding.ops, 150_000, 3
    D, I, P = _matrix(rows, cols, nnz, dtype, dev)
    B, g = torch.randn(cols, n, device=dev, dtype=D.dtype), torch.randn(rows, n, device=dev, dtype=D.dtype)
    old = ops.backward_mode()
    ops.set_backward_mode("planned")
    ops.clear_plan_cache()
    size, got = [], []
    for _ in range(4):
        got.append(ops.spdmm_backward(rows, cols, D, I, P, B, g))
        size.append(ops.plan_cache_size())
    ops.set_backward_mode(old)
    ops.clear_plan_cache()
    assert size == [0, 1, 2, 2] if want else size == [0, 1, 1, 1], size
    assert torch.equal(got[1][0], got[3][0]) and torch.equal(got[1][1], got[3][1])
    assert_close(host(got[0][0]), host(got[3][0]), "grad_A against the stateless kernels")
    assert_close(host(got[0][1]), host(got[3][1]), "grad_B against the stateless kernels")
