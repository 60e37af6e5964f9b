"""Sums of matrices with one pattern and the transpose's gradient on a symmetric one: the passes that read no
maps, at lengths around their 16 bytes a lane and with values that begin anywhere."""
import numpy as np
import pytest
import torch

import oracle
from numml_amd import _binding
from numml_amd import generators as G
from numml_amd import sparse as sp
from util import assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def eager():
    old = _binding.backward_mode()
    _binding.set_backward_mode("eager")
    yield
    _binding.set_backward_mode(old)


def _off(values, dev, by):
    """The values at `by` elements into a buffer."""
    room = torch.empty(values.size + by, dtype=torch.from_numpy(values).dtype, device=dev)
    room[by:] = torch.from_numpy(values).to(dev)
    return room[by:]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 1023, 4097])
def test_sum_and_its_gradients(dev, dtype, n):
    d, i, p, (rows, cols) = G.tridiag(n, dtype)
    d, e = randn(1, d.shape, dtype), randn(2, d.shape, dtype)
    for by in (0, 1, 3):
        I, P = to_dev(dev, i, p)
        A = sp.SparseCSRTensor((_off(d, dev, by), I, P), (rows, cols), clone=False)
        B = sp.SparseCSRTensor((_off(e, dev, by), I, P), (rows, cols), clone=False)
        A.data = A.data.detach().requires_grad_(True)
        B.data = B.data.detach().requires_grad_(True)
        g = _off(randn(3, d.shape, dtype), dev, by)
        for _ in range(2):      # (the first sum makes the plan)
            C = A - B
        ref = oracle.splincomb_forward(rows, cols, 1.0, d, i, p, -1.0, e, i, p)
        assert_same(host(C.data), ref[0], "values")
        assert_same(host(C.indices), ref[1], "columns")
        gA, gB = torch.autograd.grad(C.data, (A.data, B.data), g, retain_graph=True)
        assert_same(host(gA), host(g), "grad_A")
        assert_same(host(gB), -host(g), "grad_B")
        only, = torch.autograd.grad(C.data, (B.data,), g)
        assert torch.equal(only, gB)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_one_pattern_and_its_part(dev, dtype):
    """As many entries, but other ones: the maps are read."""
    q = np.array([0, 1, 3], np.int64)
    x, y = randn(4, 3, dtype), randn(5, 3, dtype)
    # rows (0), (0, 1) and (0), (0, 1): one pattern; rows (0), (0, 1) and (1), (0, 1): two of the same size
    for other in (np.array([0, 0, 1], np.int64), np.array([1, 0, 1], np.int64)):
        A = sp.SparseCSRTensor(tuple(to_dev(dev, x, np.array([0, 0, 1], np.int64), q)), (2, 2), clone=False)
        B = sp.SparseCSRTensor(tuple(to_dev(dev, y, other, q)), (2, 2), clone=False)
        A.requires_grad = B.requires_grad = True
        for _ in range(2):
            C = A + B
        ref = oracle.splincomb_forward(2, 2, 1.0, x, np.array([0, 0, 1], np.int64), q, 1.0, y, other, q)
        assert_same(host(C.data), ref[0], "values")
        g = randn(6, ref[0].shape, dtype)
        want = oracle.splincomb_backward(2, 2, 1.0, x, np.array([0, 0, 1], np.int64), q, 1.0, y, other, q, g, ref[1], ref[2])
        for got, w in zip(torch.autograd.grad(C.data, (A.data, B.data), to_dev(dev, g)[0]), want):
            assert_same(host(got), w, "gradient")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 40, 41])
def test_gradient_of_the_transpose(dev, dtype, n):
    cases = [G.tridiag(n, dtype), G.random_csr(n, n + 3, 0.3, 4, dtype), G.random_csr(n, n, 0.3, 5, dtype)]
    # a symmetric pattern that names an entry twice
    cases.append((randn(6, 5, dtype), np.array([0, 1, 1, 0, 0], np.int64), np.array([0, 3, 5], np.int64), (2, 2)))
    for d, i, p, (rows, cols) in cases:
        for by in (0, 1):
            I, P = to_dev(dev, i, p)
            A = sp.SparseCSRTensor((_off(d, dev, by), I, P), (rows, cols), clone=False)
            A.data = A.data.detach().requires_grad_(True)
            At = A.T
            ref = oracle.csr_transpose(rows, cols, d, i, p)
            assert_same(host(At.data), ref[0], "values")
            assert_same(host(At.indices), ref[1], "columns")
            assert_same(host(At.indptr), ref[2], "row pointers")
            g = randn(7, d.shape, dtype)
            got, = torch.autograd.grad(At.data, A.data, _off(g, dev, by))
            want = np.empty_like(g)
            want[ref[3]] = g
            assert_same(host(got), want, "gradient")
