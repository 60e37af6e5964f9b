"""Sums and products with an explicit transpose, whose structure tensors are new on every call: from the
second transpose on these are known by the plan they come from, so the pair's plan is found without a
pass over them, in the serial loop's bits."""
import numpy as np
import pytest
import torch

import numml_amd
import oracle
from numml_amd import generators as G
from numml_amd import sparse as sp
from util import assert_same, host, randn, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def ext():
    e = numml_amd.load_compiled()
    old = e.backward_mode()
    e.set_backward_mode("planned")
    e.clear_plan_cache()
    yield e
    e.set_backward_mode(old)
    e.clear_plan_cache()


def _sum_reference(r, d, i, p, g):
    td, ti, tp, back = oracle.csr_transpose(r, r, d, i, p)
    Cd, Ci, Cp = oracle.splincomb_forward(r, r, 1., d, i, p, 1., td, ti, tp)
    gA, gT = oracle.splincomb_backward(r, r, 1., d, i, p, 1., td, ti, tp, g[:Cd.size], Ci, Cp)
    gA = gA.copy()
    gA[np.asarray(back, np.int64)] += gT
    return Cd, Ci, Cp, gA


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("make", [lambda t: G.ragged_csr(700, 700, 6, 1, t), lambda t: G.poisson2d(33, t)])
def test_sum_with_the_transpose(dev, ext, dtype, make):
    d, i, p, (r, _) = make(dtype)
    i, p = np.asarray(i, np.int64), np.asarray(p, np.int64)
    I, P = to_dev(dev, i, p)
    shared = keys = None
    for call in range(6):
        v = randn(call, d.size, dtype)
        A = sp.SparseCSRTensor((to_dev(dev, v)[0], I, P), (r, r), clone=False)
        A.requires_grad = True
        C = A + A.T
        g = randn(50 + call, 2 * d.size, dtype)
        Cd, Ci, Cp, gA = _sum_reference(r, v, i, p, g)
        got, = torch.autograd.grad(C.data, A.data, to_dev(dev, g[:Cd.size])[0])
        for a, b, what in ((C.data, Cd, "data"), (C.indices, Ci, "indices"), (C.indptr, Cp, "indptr"), (got, gA, "grad")):
            assert_same(host(a), b, f"call {call} {what}")
        if call >= 4:
            assert C.indices.data_ptr() == shared and ext.plan_cache_stats()[1] == keys, f"call {call}"
        shared, keys = C.indices.data_ptr(), ext.plan_cache_stats()[1]


def test_a_pattern_edited_in_place(dev, ext):
    d, i, p, (r, _) = G.ragged_csr(300, 300, 5, 2, np.float64)
    i, p = np.asarray(i, np.int64), np.asarray(p, np.int64)
    I, P, D = to_dev(dev, i, p, d)
    A = sp.SparseCSRTensor((D, I, P), (r, r), clone=False)
    for _ in range(5):
        (A + A.T).data
    T = A.T
    # the transpose's own tensors, edited: their key is not the plan's any more.  Every row's columns are mirrored in turn,
    # so they stay sorted and distinct.
    td, ti, tp = host(T.data), host(T.indices), host(T.indptr)
    mirrored = np.concatenate([r - 1 - ti[tp[q]:tp[q + 1]][::-1] for q in range(r)])
    assert (mirrored != ti).any()
    T.indices.copy_(to_dev(dev, mirrored)[0])
    S = A + T
    Cd, Ci, Cp = oracle.splincomb_forward(r, r, 1., d, i, p, 1., td, mirrored, tp)
    for a, b in zip((S.data, S.indices, S.indptr), (Cd, Ci, Cp)):
        assert_same(host(a), b)
    # a product with it as well, and with the transpose as it was
    Cd, Ci, Cp = oracle.spgemm_forward(r, r, td, mirrored, tp, r, r, d, i, p)
    S = T @ A
    assert_same(host(S.indices), Ci)
    assert_same(host(S.data), Cd)
    T.indices.copy_(to_dev(dev, ti)[0])
    for a, b in zip((A + T).data, oracle.splincomb_forward(r, r, 1., d, i, p, 1., td, ti, tp)[0]):
        assert a == b
    # the matrix's, edited: another pattern altogether
    k = int(np.flatnonzero(np.diff(p) > 0)[0])
    row = np.repeat(np.arange(r), np.diff(p))
    i2 = i.copy()
    last = p[k + 1] - 1
    i2[last] = r - 1
    if p[k + 1] - p[k] > 1 and i[last - 1] >= i2[last]:
        i2[last] = i[last]
    I.copy_(to_dev(dev, i2)[0])
    S = A + A.T
    want = _sum_reference(r, d, i2, p, randn(1, 2 * d.size, np.float64))
    assert row.size == d.size
    for a, b in zip((S.data, S.indices, S.indptr), want):
        assert_same(host(a), b)


def test_product_with_the_transpose(dev, ext):
    n = 41
    d, i, p, (r, _) = G.poisson2d(n, np.float64)
    i, p = np.asarray(i, np.int64), np.asarray(p, np.int64)
    I, P = to_dev(dev, i, p)
    keys = None
    for call in range(6):
        v = randn(call, d.size, np.float64)
        A = sp.SparseCSRTensor((to_dev(dev, v)[0], I, P), (r, r), clone=False)
        A.requires_grad = True
        C = A.T @ A
        td, ti, tp, back = oracle.csr_transpose(r, r, v, i, p)
        Cd, Ci, Cp = oracle.spgemm_forward(r, r, td, ti, tp, r, r, v, i, p)
        assert_same(host(C.indices), Ci, f"call {call}")
        assert_same(host(C.data), Cd, f"call {call}")
        g = randn(60 + call, Cd.size, np.float64)
        got, = torch.autograd.grad(C.data, A.data, to_dev(dev, g)[0])
        gT, gA = oracle.spgemm_backward(g, Ci, Cp, r, r, td, ti, tp, r, r, v, i, p)
        gA = gA.copy()
        gA[np.asarray(back, np.int64)] += gT
        assert np.allclose(host(got), gA, rtol=1e-12, atol=1e-12 * np.abs(gA).max())
        if call >= 4:
            assert ext.plan_cache_stats()[1] == keys, f"call {call}"
        keys = ext.plan_cache_stats()[1]


@pytest.mark.parametrize("before", [1, 2, 4])
def test_in_a_graph(dev, ext, before):
    # a transpose captured as the second one of its pattern makes no key; later ones hand theirs on
    d, i, p, (r, _) = G.poisson2d(21, np.float64)
    I, P, V = to_dev(dev, np.asarray(i, np.int64), np.asarray(p, np.int64), d)
    for _ in range(before):
        ops = ext.csr_transpose_forward(r, r, V, I, P)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ext.csr_transpose_forward(r, r, V, I, P)
    for seed in (1, 2, 3):
        v = randn(seed, d.size, np.float64)
        V.copy_(torch.from_numpy(v))
        graph.replay()
        eager = ext.csr_transpose_forward(r, r, V, I, P)
        torch.cuda.synchronize()
        want = oracle.csr_transpose(r, r, v, np.asarray(i, np.int64), np.asarray(p, np.int64))
        for a, b, c in zip(out, eager, want):
            assert_same(host(a), np.asarray(c, host(a).dtype))
            assert_same(host(b), np.asarray(c, host(b).dtype))
    assert len(ops) == 4
