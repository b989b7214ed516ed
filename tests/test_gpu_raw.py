"""Multivector memory as it lies in HBM, read and written through the handle's
data pointer by copies of the runtime's default stream: what a call has written
is there, for other streams than the library's, when it returns its numbers."""
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
    return lib


def raw(mv):
    """All of a multivector's memory, padding rows included: (ld, ncols)."""
    h = Handle.from_address(mv.ptr)
    out = np.empty((h.ld, h.ncols), dtype=np.float64 if h.prec == F64 else np.float32, order="F")
    assert hip().hipMemcpy(out.ctypes.data, h.data, out.nbytes, 2) == 0
    return out


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
