"""Host columns into and out of multivectors of an ordered matrix and of FP32
ones, in one go and in several (a block larger than the device staging buffer),
and gradients whose Jacobian indices go through the entry order or are bad."""
import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, capi, eig_gradient
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("m,k", [(1, 1), (17, 3), (1101, 9)])
def test_columns_round_trip(m, k, prec, ordered):
    A = P.lap2d(m)[0]
    n, g = m * m, np.random.default_rng(m)
    perm = g.permutation(n).astype(np.int32) if ordered else None
    mat = Matrix(A, order=perm)
    X = np.asfortranarray(g.standard_normal((n, k)))
    mv = MultiVec(mat, k, prec)
    mv.set(X)
    want = X if prec == F64 else X.astype(np.float32).astype(np.float64)
    assert np.array_equal(mv.get(), want)
    # a host block with rows and columns to spare, which stay as they are
    H = np.full((n + 5, k + 2), 7.0, order="F")
    capi.load().HIP_MultiVecGetToHost(mv.ptr, 0, k, H[:, 1:].ctypes.data_as(capi.DP), n + 5)
    capi.raise_on_error("get")
    assert np.array_equal(H[:n, 1:k + 1], want) and np.all(H[n:] == 7.0) and np.all(H[:, [0, k + 1]] == 7.0)
    H[:n, 1:k + 1] *= 2.0
    capi.load().HIP_MultiVecSetFromHost(mv.ptr, k - 1, 1, H[:, 1:].ctypes.data_as(capi.DP), n + 5)
    capi.raise_on_error("set")
    want = want.copy()
    want[:, k - 1] = H[:n, 1]
    assert np.array_equal(mv.get(), want)


def test_gradient_order_and_bad_indices():
    A = P.lap2d(24)[0]
    n, k, g = A.shape[0], 3, np.random.default_rng(1)
    X, w = np.asfortranarray(g.standard_normal((n, k))), g.uniform(0.5, 2.0, k)
    jrp = np.concatenate([[0], np.cumsum(g.integers(0, 9, 300))]).astype(np.int32)
    jnz = g.integers(0, A.nnz, jrp[-1]).astype(np.int32)
    jval = g.standard_normal(jrp[-1])
    args = (w, 300, jrp, jnz, jval)
    natural, ordered = Matrix(A), Matrix(A, order=g.permutation(n).astype(np.int32))
    want = eig_gradient(natural, X, *args)
    # the same products in the same order, entry by entry
    assert np.array_equal(eig_gradient(ordered, X, *args), want)
    for at, value in ((0, -1), (len(jnz) - 1, A.nnz)):
        bad = jnz.copy()
        bad[at] = value
        for mat in (natural, ordered):
            with pytest.raises(Exception, match=r"jnz\[%d\]=%d" % (at, value)):
                eig_gradient(mat, X, w, 300, jrp, bad, jval)
    assert np.array_equal(eig_gradient(ordered, X, *args), want)
