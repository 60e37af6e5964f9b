"""Differentiable sparse triangular solve, and the direct solve built on it: LU without
pivoting followed by two triangular solves (numml/sparse/linalg.py:8-137)."""
import torch

from .._binding import ops as _ext
from ._csr import _native

__all__ = ["sptrsv", "spsolve_triangular", "splu", "splu_solve", "spsolve_fn", "spsolve"]


class sptrsv(torch.autograd.Function):
    """x = A^{-1} b for a triangular CSR matrix with a single right-hand side.

    Gradients: grad_b = A^{-T} grad_x and grad_A[k] = -grad_b[row] x[col] on every
    stored entry (cpp/sparse_csr_cpu.cpp:725-759).
    """

    @staticmethod
    def forward(ctx, shape, A_data, A_indices, A_indptr, lower, unit, b):
        if shape[0] != shape[1]:
            raise RuntimeError(
                f"Expected square matrix for triangular solve, got {shape[0]} x {shape[1]}.")
        if A_data.type() != b.type():
            raise RuntimeError("Matrix and vector should be same data type, got "
                               f"{A_data.type()} and {b.type()}, respectively.")
        x = _ext.sptrsv_forward(shape[0], shape[1], A_data, A_indices, A_indptr, lower, unit, b)
        ctx.save_for_backward(A_data, A_indices, A_indptr, b, x)
        ctx.lower, ctx.unit, ctx.shape = lower, unit, shape
        return x

    @staticmethod
    def backward(ctx, grad_x):
        A_data, A_indices, A_indptr, b, x = ctx.saved_tensors
        grad_A, grad_b = _ext.sptrsv_backward(grad_x, x, ctx.shape[0], ctx.shape[1], A_data,
                                              A_indices, A_indptr, ctx.lower, ctx.unit, b)
        return None, grad_A, None, None, None, None, grad_b


def spsolve_triangular(A, b, lower=True, unit_diagonal=False):
    """Solve A x = b for triangular A (numml/sparse/linalg.py:116-137)."""
    if _native(A.data, b) and A.shape[0] == A.shape[1]:
        return _ext.sptrsv_node(A.shape[0], A.data, A.indices, A.indptr, lower, unit_diagonal, b)
    return sptrsv.apply(A.shape, A.data, A.indices, A.indptr, lower, unit_diagonal, b)


def splu(A):
    """Sparse LU factorisation of an invertible matrix, without pivoting: the result holds
    L (unit diagonal, not stored) below and U on and above the diagonal, on the pattern of A
    plus its fill.  Carries no gradient; use spsolve for a differentiable solve
    (numml/sparse/linalg.py:47-56)."""
    from ._csr import SparseCSRTensor
    M_data, M_indices, M_indptr = _ext.splu(A.shape[0], A.shape[1], A.data, A.indices, A.indptr)[:3]
    return SparseCSRTensor((M_data, M_indices, M_indptr), A.shape)


def splu_solve(A_LU, b):
    """Solve A x = b given A_LU = splu(A) (numml/sparse/linalg.py:62-79)."""
    y = spsolve_triangular(A_LU, b, True, True)
    return spsolve_triangular(A_LU, y, False, False)


class spsolve_fn(torch.autograd.Function):
    """x = A^{-1} b by LU.  Gradients: grad_b = A^{-T} grad_x through the transposed factors,
    grad_A[k] = -grad_b[row] x[col] on A's stored entries (numml/sparse/linalg.py:82-110)."""

    @staticmethod
    def forward(ctx, A_shape, A_data, A_indices, A_indptr, b):
        M_data, M_indices, M_indptr, Mt_data, Mt_indices, Mt_indptr = \
            _ext.splu(A_shape[0], A_shape[1], A_data, A_indices, A_indptr)
        y = _ext.sptrsv_forward(A_shape[0], A_shape[1], M_data, M_indices, M_indptr, True, True, b)
        x = _ext.sptrsv_forward(A_shape[0], A_shape[1], M_data, M_indices, M_indptr, False, False, y)
        ctx.shape = A_shape
        ctx.save_for_backward(A_data, A_indices, A_indptr, Mt_data, Mt_indices, Mt_indptr, x)
        return x

    @staticmethod
    def backward(ctx, grad_x):
        A_data, A_indices, A_indptr, Mt_data, Mt_indices, Mt_indptr, x = ctx.saved_tensors
        grad_A, grad_b = _ext.spsolve_backward(grad_x, x, ctx.shape[0], ctx.shape[1], Mt_data, Mt_indices,
                                               Mt_indptr, A_data, A_indices, A_indptr)
        return None, grad_A, None, None, grad_b


def spsolve(A, b):
    """Solve A x = b for a general sparse A (numml/sparse/linalg.py:113-114)."""
    if _native(A.data, b) and A.shape[0] == A.shape[1]:
        return _ext.spsolve_node(A.shape[0], A.data, A.indices, A.indptr, b)
    return spsolve_fn.apply(A.shape, A.data, A.indices, A.indptr, b)
