"""Staged row blocks on grids: bricks of a lexicographically numbered box grid
(the default for its natural order), consecutive rows of a tile order, rows of
up to 28 entries held in registers and longer ones beside them, and the
residual check that stages X once for A and B.  Products are bit-identical to
the oracle's CSR loop; reductions differ in summation order only."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle_api as O
from gcge_hip import Matrix, MultiVec, Ops, capi
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32


def stencil(shape, reach, seed):
    """Random symmetric-pattern stencil on a box (last axis fastest): all
    offsets within `reach` (a set of offset sums of squares)."""
    r = np.random.default_rng(seed)
    idx = np.arange(np.prod(shape)).reshape(shape)
    rows, cols = [], []
    for off in np.ndindex(*(3,) * len(shape)):
        o = np.array(off) - 1
        if int(np.sum(o * o)) not in reach:
            continue
        a = tuple(slice(max(0, -d), s - max(0, d)) for d, s in zip(o, shape))
        b = tuple(slice(max(0, d), s + min(0, d)) for d, s in zip(o, shape))
        rows.append(idx[a].ravel())
        cols.append(idx[b].ravel())
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    M = sp.csr_matrix((r.standard_normal(rows.size), (rows, cols)), shape=(idx.size, idx.size))
    M.sort_indices()
    M.indptr, M.indices = M.indptr.astype(np.int32), M.indices.astype(np.int32)
    return M


# 7- and 27-point stencils on boxes whose extents no brick divides, one brick
# in x, several in every direction, a 3-D box beyond 500,000 cells with odd
# lines (consecutive rows), and 2-D boxes (5- and 9-point)
CASES = {"7pt": ((19, 21, 37), {0, 1}), "27pt": ((19, 21, 37), {0, 1, 2, 3}), "7pt_thin": ((40, 33, 6), {0, 1}),
         "27pt_long": ((5, 9, 300), {0, 1, 2, 3}), "7pt_plane": ((61, 92, 91), {0, 1}), "27pt_plane": ((61, 92, 91), {0, 1, 2, 3}), "5pt": ((70, 131), {0, 1}), "9pt": ((70, 131), {0, 1, 2})}


@pytest.fixture(scope="module")
def ops():
    o = Ops()
    yield o
    o.close()


@pytest.mark.parametrize("order", [None, "locality"])
@pytest.mark.parametrize("name", list(CASES))
def test_staged_spmm(ops, name, order):
    A = stencil(*CASES[name], seed=1)
    n = A.shape[0]
    mA = Matrix(A, order=order)
    assert capi.load().HIP_MatGatherKind(mA.ptr) == 2
    for k in (1, 4, 7, 130) if n < 100000 else (7,):
        X = np.random.default_rng(k).standard_normal((n, k))
        Y = O.csr_matmultivec(A, X)
        x, y, z = MultiVec(mA, k, data=X), MultiVec(mA, k), MultiVec(mA, k)
        ops.matdot(mA, x, y)
        np.testing.assert_array_equal(y.get(), Y)
        d = ops.matdot_dot(mA, x, z)
        np.testing.assert_array_equal(z.get(), Y)
        # |sum| of k-term products in another order: n eps of the sum of magnitudes
        np.testing.assert_array_less(np.abs(d - np.einsum("ij,ij->j", X, Y)),
                                     1e-13 * np.einsum("ij,ij->j", np.abs(X), np.abs(Y)))
        xf, yf = MultiVec(mA, k, F32, data=X), MultiVec(mA, k, F32)
        ops.matdot(mA, xf, yf)
        A32, X32 = A.astype(np.float32).astype(np.float64), X.astype(np.float32).astype(np.float64)
        bound = 28 * 2.0 ** -23 * (abs(A32) @ np.abs(X32))
        assert np.all(np.abs(yf.get() - A32 @ X32) <= bound)
        for m in (x, y, z, xf, yf):
            m.close()
    mA.close()


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("pair", [("7pt", None), ("27pt", None), ("7pt", "27pt"), ("27pt", "7pt"), ("27pt", "27pt"),
                                  ("7pt", "7pt"), ("5pt", "9pt"), ("7pt_plane", "27pt_plane"), ("7pt_plane", None)])
@pytest.mark.parametrize("order", [None, "locality"])
def test_staged_residual(ops, prec, pair, order):
    A = stencil(*CASES[pair[0]], seed=2)
    B = stencil(*CASES[pair[1]], seed=3) if pair[1] else None
    n, k = A.shape[0], 9
    mA = Matrix(A, order=order)
    mB = Matrix(B, order=mA.order()) if B is not None else None
    X = np.random.default_rng(4).standard_normal((n, k + 2))
    idx = np.random.default_rng(5).permutation(k + 2)[:k].astype(np.int32)
    lam = np.random.default_rng(6).uniform(0.1, 3.0, k)
    x = MultiVec(mA, k + 2, prec, data=X)
    rn, xn, bn = ops.residual_norms(mA, mB, x, idx, lam)
    if prec == F32:
        X = X.astype(np.float32).astype(np.float64)
    X = X[:, idx]
    BX = X if B is None else B @ X
    np.testing.assert_allclose(rn, np.linalg.norm(A @ X - BX * lam, axis=0), rtol=1e-12)
    np.testing.assert_allclose(xn, np.linalg.norm(X, axis=0), rtol=1e-12)
    np.testing.assert_allclose(bn, np.linalg.norm(BX, axis=0), rtol=1e-12)


def test_staged_values_follow_updates(ops):
    """HIP_MatSetValues on a brick matrix: the products use the new values."""
    A = stencil((19, 21, 37), {0, 1}, 7)
    mA = Matrix(A)
    X = np.random.default_rng(8).standard_normal((A.shape[0], 3))
    x, y = MultiVec(mA, 3, data=X), MultiVec(mA, 3)
    A.data = np.random.default_rng(9).standard_normal(A.nnz)
    mA.set_values(A.data)
    ops.matdot(mA, x, y)
    np.testing.assert_array_equal(y.get(), O.csr_matmultivec(A, X))


def test_long_rows_stay_gathered(ops):
    """More than 28 entries per row on average: row gather as before."""
    M = sp.diags([np.ones(600 - abs(o)) for o in range(-20, 21)], range(-20, 21), format="csr")
    M.indptr, M.indices = M.indptr.astype(np.int32), M.indices.astype(np.int32)
    mM = Matrix(M)
    assert capi.load().HIP_MatGatherKind(mM.ptr) == 1
    X = np.random.default_rng(10).standard_normal((600, 5))
    x, y = MultiVec(mM, 5, data=X), MultiVec(mM, 5)
    ops.matdot(mM, x, y)
    np.testing.assert_array_equal(y.get(), O.csr_matmultivec(M, X))
