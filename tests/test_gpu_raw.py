"""Multivector memory as it lies in HBM, read and written through the handle's
data pointer by copies of the runtime's default stream: what a call has written
is there, for other streams than the library's, when it returns its numbers, and
the padding rows between a column's end and the next column keep their bits."""
import ctypes

import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, Ops, capi, synchronize
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32


class Handle(ctypes.Structure):
    """Head of a multivector handle's struct."""
    _fields_ = [("magic", ctypes.c_uint32), ("prec", ctypes.c_int), ("n", ctypes.c_int64), ("ld", ctypes.c_int64),
                ("ncols", ctypes.c_int), ("data", ctypes.c_void_p)]


def hip():
    """The HIP runtime that the library runs on (its dependencies' symbols)."""
    lib = ctypes.CDLL(capi.LIB_PATH)
    lib.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    lib.hipMemcpy2D.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t,
                                ctypes.c_size_t, ctypes.c_int]
    return lib


def raw(mv):
    """All of a multivector's memory, padding rows included: (ld, ncols)."""
    h = Handle.from_address(mv.ptr)
    out = np.empty((h.ld, h.ncols), dtype=np.float64 if h.prec == F64 else np.float32, order="F")
    assert hip().hipMemcpy(out.ctypes.data, h.data, out.nbytes, 2) == 0
    return out


NAN = {F64: 0x7ff8dead0000beef, F32: 0x7fc0dead}


def padded(mat, X, prec):
    """X as a multivector whose padding rows hold a NaN of known bits."""
    mv = MultiVec(mat, X.shape[1], prec)
    h = Handle.from_address(mv.ptr)
    T, U = (np.float64, np.uint64) if prec == F64 else (np.float32, np.uint32)
    H = np.full((h.ld, h.ncols), NAN[prec], dtype=U, order="F").view(T)
    H[:h.n] = X
    synchronize()
    assert hip().hipMemcpy(h.data, H.ctypes.data, H.nbytes, 1) == 0
    return mv


def padding_kept(mv):
    """Whether the padding rows still hold padded()'s bits."""
    h = Handle.from_address(mv.ptr)
    w, U = (8, np.uint64) if h.prec == F64 else (4, np.uint32)
    out = np.empty((h.ld - h.n, h.ncols), dtype=U, order="F")
    synchronize()
    assert hip().hipMemcpy2D(out.ctypes.data, w * (h.ld - h.n), h.data + w * h.n, w * h.ld, w * (h.ld - h.n), h.ncols,
                             2) == 0
    return bool(np.all(out == NAN[h.prec]))


@pytest.fixture(scope="module")
def ops():
    o = Ops()
    yield o
    o.close()


@pytest.mark.parametrize("prec", [F64, F32])
@pytest.mark.parametrize("m,k", [(20, 1), (128, 20), (300, 7)])
def test_columns_are_there_for_another_stream(ops, m, k, prec):
    A, g = Matrix(P.lap2d(m)[0]), np.random.default_rng(m)
    x, r, w, p = (MultiVec(A, k, prec) for _ in range(4))
    for v in (x, r, w, p):
        v.set(np.asfortranarray(g.standard_normal((m * m, k))))
    a = g.uniform(0.1, 1.0, k)
    for f, v in ((lambda: ops.matdot_dot(A, x, w), w), (lambda: ops.cg_residual_update(w, r, k, a), r),
                 (lambda: ops.pcg_residual_update(A, w, r, k, a), r),
                 (lambda: ops.cg_update(x, 0, p, w, r, k, a), r)):
        synchronize()
        f()
        seen = raw(v)
        synchronize()
        assert np.array_equal(seen[:m * m], v.get())


@pytest.mark.parametrize("prec", [F64, F32])
# one row, rows on both sides of a 16-byte access and of a 256-row block, and
# columns that the streams write past the caches
@pytest.mark.parametrize("m,k", [(1, 2), (15, 3), (16, 20), (37, 7), (1101, 42)])
def test_padding_keeps_its_bits(ops, prec, m, k):
    M = P.lap2d(m)[0]
    A, g, n = Matrix(M), np.random.default_rng(m), m * m
    other = F32 if prec == F64 else F64
    X = {c: g.integers(-4, 5, (n, k)).astype(np.float64) for c in "xprw"}
    v = {c: padded(A, X[c], prec) for c in X}
    one, a = np.ones(k), np.full(k, 2.0)

    def same(c, want):
        assert np.array_equal(v[c].get(), want), c
        assert all(padding_kept(mv) for mv in v.values())
        X[c] = want

    ops.axpby(2.0, v["x"], 1.0, v["w"])
    same("w", 2.0 * X["x"] + X["w"])
    ops.axpby(0.0, v["x"], -1.0, v["w"])
    same("w", -X["w"])
    ops.axpby_diag(one, v["p"], 0.0 * one, v["w"])
    same("w", X["p"])
    ops.copy(v["r"], v["w"])
    same("w", X["r"])
    to = padded(A, X["x"], other)
    ops.copy(v["p"], to)
    ops.copy(to, v["w"])
    same("w", X["p"])
    assert padding_kept(to)
    ops.matdot(A, v["x"], v["w"])
    same("w", M @ X["x"])
    ops.matdot_dot(A, v["p"], v["w"])
    same("w", M @ X["p"])
    ops.cg_residual_update(v["w"], v["r"], k, a)
    same("r", X["r"] - 2.0 * X["w"])
    ops.pcg_residual_update(A, v["w"], v["r"], k, a)
    same("r", X["r"] - 2.0 * X["w"])
    ops.cg_search_update(v["x"], 0, v["p"], v["r"], k, k, a, one)
    X["x"] = X["x"] + 2.0 * X["p"]
    same("p", X["r"] + X["p"])
    same("x", X["x"])
    ops.pcg_search_update(A, v["x"], 0, v["p"], v["r"], k, k, a, one)
    X["x"] = X["x"] + 2.0 * X["p"]
    same("p", 0.25 * X["r"] + X["p"])  # the diagonal is 4
    same("x", X["x"])
    ops.cg_update(v["x"], 0, v["p"], v["w"], v["r"], k, a)
    X["x"] = X["x"] + 2.0 * X["p"]
    same("r", X["r"] - 2.0 * X["w"])
    same("x", X["x"])

