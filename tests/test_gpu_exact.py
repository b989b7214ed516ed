"""Sums that are exact in any order, so that a row left out or taken twice shows:
Gram products of small integers (FP32 partial sums stay below 2^24) at every
variant of the tilings, with several row slabs per chunk and NaN in the padding
rows of both precisions, and products with few columns of a 27-point matrix."""
import ctypes

import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, Ops, capi
from gcge_hip import problems as P
from test_gpu_raw import padded

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32
ROWS = {1: 1, 1369: 37, 16900: 130, 39601: 199, 99856: 316, 140625: 375}  # rows: side of the 2-D grid


@pytest.fixture(scope="module")
def ops():
    o = Ops()
    yield o
    o.close()


@pytest.fixture(scope="module")
def mats():
    return {n: Matrix(P.lap2d(m)[0]) for n, m in ROWS.items()}


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("n", list(ROWS))
# the kernel without LDS, the thin one, and the slabs: few columns, 16 tiles
# together, 28, past 256 columns
@pytest.mark.parametrize("p,q,sym", [(32, 32, False), (4, 8, False), (50, 50, True), (64, 64, False), (40, 70, False),
                                     (130, 100, False), (100, 100, True), (200, 100, False), (200, 200, True),
                                     (300, 100, False), (289, 289, True)])
def test_gram_exact(ops, mats, prec, n, p, q, sym):
    g = np.random.default_rng(n + p * q)
    V = g.integers(-3, 4, (n, p)).astype(np.float64)
    W = V if sym else g.integers(-3, 4, (n, q)).astype(np.float64)
    v = padded(mats[n], V, prec)
    w = v if sym else padded(mats[n], W, prec)
    assert np.array_equal(ops.gram(v, w, sym=sym), V.T @ W)


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("n", [1369, 140625])
@pytest.mark.parametrize("p,q,beta", [(300, 97, 1.0), (129, 17, -2.0), (70, 113, 0.0), (63, 32, 1.0), (7, 8, 0.0)])
def test_lincomb_exact(ops, mats, prec, n, p, q, beta):
    g = np.random.default_rng(p * q)
    X, Y, C = (g.integers(-3, 4, s).astype(np.float64) for s in ((n, p), (n, q), (p, q)))
    x, y = padded(mats[n], X, prec), padded(mats[n], Y, prec)
    ops.lincomb(x, y, C, alpha=-1.0, beta=beta)
    assert np.array_equal(y.get(), -(X @ C) + (beta * Y if beta else 0.0))


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("n", [1, 1369, 39601, 99856])
# few columns into many, on both sides of the choice between the two kernels
@pytest.mark.parametrize("p,q,beta", [(1, 300, 0.0), (3, 200, 1.0), (12, 128, -1.0), (20, 48, 1.0), (25, 65, 0.0),
                                      (64, 64, 1.0), (20, 120, 0.0), (99, 113, 2.0)])
def test_lincomb_of_few_into_many(ops, mats, prec, n, p, q, beta):
    test_lincomb_exact(ops, mats, prec, n, p, q, beta)


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("order", [None, "locality"])
def test_few_columns_of_27_points(ops, prec, k, order):
    M = P.lap3d_mass(19)[1]
    g = np.random.default_rng(k)
    M.data = g.integers(-3, 4, M.nnz).astype(np.float64)
    A = Matrix(M, order=order)
    X = g.integers(-3, 4, (M.shape[0], k)).astype(np.float64)
    Y = M @ X
    x, y = MultiVec(A, k, prec, data=X), MultiVec(A, k, prec)
    ops.matdot(A, x, y)
    assert np.array_equal(y.get(), Y)
    assert np.array_equal(ops.matdot_dot(A, x, y), np.sum(X * Y, axis=0)) and np.array_equal(y.get(), Y)
    lam = g.integers(-2, 3, k).astype(np.float64)
    for B, BX in ((None, X), (A, Y)):
        rn, xn, bn = ops.residual_norms(A, B, x, np.arange(k), lam)
        R = Y - BX * lam
        assert np.array_equal(np.stack([rn, xn, bn]), np.sqrt(np.stack([np.sum(v * v, axis=0) for v in (R, X, BX)])))
