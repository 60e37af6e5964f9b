"""Gradients around the Functions that return structure beside values: scalars of a linear combination,
and a gradient of the values that is missing (counts as zeros)."""
import numpy as np
import pytest
import torch

from numml_amd import generators as G
from numml_amd import sparse as sp
from util import host, to_dev

pytestmark = pytest.mark.gpu


class _NoGradient(torch.autograd.Function):
    """Passes its input on and hands no gradient back."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, _g):
        return None


def _matrix(dev):
    d, i, p, shape = G.poisson2d(9, np.float64)
    d = d * np.random.default_rng(3).uniform(1, 2, d.size)
    A = sp.SparseCSRTensor(tuple(to_dev(dev, d, i, p)), shape, clone=False)
    A.requires_grad = True
    return A


def test_scalars_of_a_linear_combination(dev):
    A, B = _matrix(dev), _matrix(dev)
    alpha = torch.tensor(2.0, dtype=torch.float64, requires_grad=True)
    beta = torch.tensor(-3.0, dtype=torch.float64)
    C, _, _ = sp._csr.splincomb.apply(A.shape, alpha, A.data, A.indices, A.indptr, beta, B.data, B.indices, B.indptr)
    g_alpha, g_A, g_B = torch.autograd.grad(C.sum(), (alpha, A.data, B.data))
    assert np.isclose(host(g_alpha), host(A.data).sum(), rtol=1e-12)
    assert np.array_equal(host(g_A), np.full(A.nnz, 2.0)) and np.array_equal(host(g_B), np.full(B.nnz, -3.0))


@pytest.mark.parametrize("make", [lambda A: (A @ A).data, lambda A: A.T.data, lambda A: (A + A).data])
def test_missing_gradient_counts_as_zeros(dev, make):
    A = _matrix(dev)
    (_NoGradient.apply(make(A)).sum() + A.data.sum()).backward()
    assert np.array_equal(host(A.data.grad), np.ones(A.nnz))
