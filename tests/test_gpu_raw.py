"""Multivector memory as it lies in HBM, read and written by torch through the
handle's data pointer: what a call has written is there for another stream
when the call returns its numbers."""
import ctypes
import types

import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, Ops, capi, synchronize
from gcge_hip import problems as P

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32


class Handle(ctypes.Structure):
    """Head of a multivector handle's struct."""
    _fields_ = [("magic", ctypes.c_uint32), ("prec", ctypes.c_int), ("n", ctypes.c_int64), ("ld", ctypes.c_int64),
                ("ncols", ctypes.c_int), ("data", ctypes.c_void_p)]


def raw(mv):
    """All of a multivector's memory, padding rows included, as an (ncols, ld)
    tensor without a copy."""
    h = Handle.from_address(mv.ptr)
    w = 8 if h.prec == F64 else 4
    iface = dict(shape=(h.ncols, h.ld), typestr="<f%d" % w, data=(h.data, False), version=3, strides=None)
    return torch.as_tensor(types.SimpleNamespace(__cuda_array_interface__=iface, owner=mv), device="cuda")


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
    other = torch.cuda.Stream()
    for f, v in ((lambda: ops.matdot_dot(A, x, w), w), (lambda: ops.cg_residual_update(w, r, k, a), r),
                 (lambda: ops.pcg_residual_update(A, w, r, k, a), r),
                 (lambda: ops.cg_update(x, 0, p, w, r, k, a), r)):
        mem = raw(v)
        f()
        with torch.cuda.stream(other):
            seen = mem.clone()
        other.synchronize()
        synchronize()
        assert torch.equal(seen[:, :m * m].double().cpu(), torch.from_numpy(v.get().T.copy()))
