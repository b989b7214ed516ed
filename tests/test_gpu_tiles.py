"""Block combinations and Gram products at the edges of their tilings: row
counts on both sides of each rows-per-wavefront choice, none a multiple of a
tile, one to several passes of column blocks, partial last k blocks, and
multivectors whose padding rows hold NaN (a host block with the device's
leading dimension brings its own padding along).  Reference: FP64 products of
the stored values; the bounds are the rounding of a sum of p (or n) terms."""
import ctypes as C

import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, Ops, capi
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32
ROWS = {1369: 37, 99856: 316, 140625: 375}  # rows: side of the 2-D grid
EPS = {F64: 2.0 ** -53, F32: 2.0 ** -24}


@pytest.fixture(scope="module")
def ops():
    o = Ops()
    yield o
    o.close()


@pytest.fixture(scope="module")
def mats():
    return {n: Matrix(P.lap2d(m)[0]) for n, m in ROWS.items()}


def nan_padded(mat, X, prec):
    """X (FP64: through a host block with the device's leading dimension, NaN
    below its n rows)."""
    n, k = X.shape
    mv = MultiVec(mat, k, prec)
    if prec == F64:
        ld = ((n + 255) // 256 | 1) * 256
        H = np.full((ld, k), np.nan, order="F")
        H[:n] = X
        capi.load().HIP_MultiVecSetFromHost(mv.ptr, 0, k, H.ctypes.data_as(capi.DP), ld)
        capi.raise_on_error("set")
    else:
        mv.set(X)
    return mv


def stored(X, prec):
    return X if prec == F64 else X.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("n", list(ROWS))
@pytest.mark.parametrize("p,q,alpha,beta", [(130, 100, 1.0, 0.0), (301, 97, -1.0, 1.0), (129, 17, 0.5, -2.0),
                                            (70, 113, 1.0, 0.0), (255, 130, -1.0, 1.0), (63, 32, 1.0, 0.0),
                                            (64, 33, 1.0, 1.0), (2, 65, 1.0, 0.0)])
def test_lincomb_edges(ops, mats, prec, n, p, q, alpha, beta):
    g = np.random.default_rng(p * q)
    X, Y, cf = g.standard_normal((n, p)), g.standard_normal((n, q)), g.standard_normal((p, q))
    x, y = nan_padded(mats[n], X, prec), nan_padded(mats[n], Y, prec)
    ops.lincomb(x, y, cf, alpha=alpha, beta=beta)
    X, Y, cf = stored(X, prec), stored(Y, prec), stored(cf, prec)
    ref = alpha * (X @ cf) + (beta * Y if beta else 0.0)
    bound = (p + 3) * EPS[prec] * (abs(alpha) * (np.abs(X) @ np.abs(cf)) + abs(beta) * np.abs(Y))
    assert np.all(np.abs(y.get() - ref) <= bound)


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("n", list(ROWS))
@pytest.mark.parametrize("p,q,sym", [(33, 48, False), (16, 65, False), (81, 3, False), (300, 97, False),
                                     (128, 128, False), (129, 130, False), (351, 100, False), (449, 17, False),
                                     (33, 33, True), (49, 49, True), (100, 100, True), (129, 129, True),
                                     (289, 289, True)])
def test_gram_edges(ops, mats, prec, n, p, q, sym):
    if n * (p + q) > 6.0e7:
        pytest.skip("host reference too long")
    g = np.random.default_rng(p * q + sym)
    V = g.standard_normal((n, p))
    W = V if sym else g.standard_normal((n, q))
    v = nan_padded(mats[n], V, prec)
    w = v if sym else nan_padded(mats[n], W, prec)
    G = ops.gram(v, w, sym=sym)
    V, W = stored(V, prec), stored(W, prec)
    err = np.abs(G - V.T @ W)
    # the device's sum of n terms, and the host's in FP64
    bound = (n + 1) * (EPS[prec] + EPS[F64]) * (np.abs(V).T @ np.abs(W))
    if sym:
        err = np.triu(err)
    assert np.all(err <= bound)
