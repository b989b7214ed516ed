"""Element-wise kernels and their dots at the edges of 16-byte accesses (row
counts that no access divides, one row, padding rows that hold NaN) and with
blocks on both sides of the size from which they bypass the caches.  Element by
element every result is the rounding of each product and each sum, so bits are
compared; a dot of n terms may differ by n roundings of its absolute sum."""
import numpy as np
import pytest

from gcge_hip import Matrix, MultiVec, Ops, capi
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32
TYPE = {F64: np.float64, F32: np.float32}


@pytest.fixture(scope="module")
def ops():
    o = Ops()
    yield o
    o.close()


@pytest.mark.parametrize("m,k,prec", [(1, 1, F64), (1, 2, F32), (3, 5, F32), (37, 3, F64), (37, 130, F32),
                                      (1025, 2, F64), (1025, 2, F32), (1101, 20, F64), (1101, 41, F32)])
def test_streams(ops, m, k, prec):
    A, T = Matrix(P.lap2d(m)[0]), TYPE[prec]  # diagonal 4: its inverse is exact
    n, g = m * m, np.random.default_rng(m + k)
    host = {c: g.standard_normal((n, k)).astype(T) for c in "xpr"}
    dev = {c: MultiVec(A, k, prec) for c in "xprw"}
    for c in "xpr":
        dev[c].set(np.asfortranarray(host[c], dtype=np.float64))
    x, p, r = (host[c] for c in "xpr")
    al, be = g.uniform(0.1, 2.0, k), g.uniform(0.1, 2.0, k)
    a, b = al.astype(T), be.astype(T)

    ops.copy(dev["p"], dev["w"])
    assert np.array_equal(dev["w"].get(), p)
    ops.axpby_diag(al, dev["r"], be, dev["w"])
    w = a * r + b * p
    assert np.array_equal(dev["w"].get(), w)
    ops.axpby(0.0, dev["r"], 0.5, dev["w"])
    assert np.array_equal(dev["w"].get(), T(0.5) * w)
    ops.axpby(-2.0, dev["p"], 0.0, dev["w"])
    w = T(-2.0) * p
    assert np.array_equal(dev["w"].get(), w)

    def close(got, u, v):
        u, v = u.astype(np.float64), v.astype(np.float64)
        bound = (n + 1) * 2.0 ** -53 * 2.0 * np.sum(np.abs(u * v), axis=0)
        assert np.all(np.abs(got - np.sum(u * v, axis=0)) <= bound)

    close(ops.dots(dev["x"], dev["r"]), x, r)
    close(ops.cg_residual_update(dev["w"], dev["r"], k, al), *(2 * [(r := r - a * w)]))
    rz, rr = ops.pcg_residual_update(A, dev["w"], dev["r"], k, be)
    r = r - b * w
    assert np.array_equal(dev["r"].get(), r)
    close(rz, r, r * T(0.25))
    close(rr, r, r)
    kx, kp = k, (k + 1) // 2  # fewer search directions than solutions
    ops.pcg_search_update(A, dev["x"], 0, dev["p"], dev["r"], kx, kp, al, be)
    x = x + a * p
    p[:, :kp] = r[:, :kp] * T(0.25) + b[:kp] * p[:, :kp]
    assert np.array_equal(dev["x"].get(), x) and np.array_equal(dev["p"].get(), p)
    ops.cg_search_update(dev["x"], 0, dev["p"], dev["r"], kp, kx, al, be)
    x[:, :kp] = x[:, :kp] + a[:kp] * p[:, :kp]
    p = r + b * p
    assert np.array_equal(dev["x"].get(), x) and np.array_equal(dev["p"].get(), p)


def test_copy_converts_and_keeps_padding(ops):
    A = Matrix(P.lap2d(37)[0])
    n, k, ld = 1369, 7, (1369 // 256 + 1 | 1) * 256
    H = np.full((ld, k), np.nan, order="F")
    H[:n] = np.random.default_rng(5).standard_normal((n, k))
    x, f, y = MultiVec(A, k, F64), MultiVec(A, k, F32), MultiVec(A, k, F64)
    capi.load().HIP_MultiVecSetFromHost(x.ptr, 0, k, H.ctypes.data_as(capi.DP), ld)
    capi.raise_on_error("set")
    ops.copy(x, f, xs=1, ys=2, k=5)
    ops.copy(f, y, xs=2, ys=0, k=5)
    assert np.array_equal(y.get()[:, :5], H[:n, 1:6].astype(np.float32).astype(np.float64))


def test_few_partial_sums(ops):
    """8 columns of 256 blocks are added on the host, 9 on the device, in one
    order; a NaN with the bits that mark a sum as not there yet ends in NaN."""
    A = Matrix(P.lap2d(300)[0])
    n, g = 90000, np.random.default_rng(3)
    x, y = MultiVec(A, 9, F64), MultiVec(A, 9, F64)
    X = np.asfortranarray(g.standard_normal((n, 9)))
    x.set(X)
    y.set(np.asfortranarray(g.standard_normal((n, 9))))
    nine = ops.dots(x, y)
    assert np.array_equal(ops.dots(x, y, 8), nine[:8])
    assert np.array_equal(ops.dots(x, y, 1), nine[:1])
    X[5, 3] = np.array([0x7ff5a3c96e1d8b47], dtype=np.uint64).view(np.float64)[0]
    X[6, 4] = np.array([0x7ffda3c96e1d8b47], dtype=np.uint64).view(np.float64)[0]
    x.set(X)
    got = ops.dots(x, y, 8)
    assert np.all(np.isnan(got) == [False] * 3 + [True] * 2 + [False] * 3)
    got[3:5] = nine[3:5]
    assert np.array_equal(got, nine[:8])


@pytest.mark.parametrize("p,q", [(16, 126), (64, 32), (65, 33), (9, 9), (331, 129)])
def test_staged_coefficients(ops, p, q):
    """Coefficients on both sides of the size from which a kernel fetches them,
    several launches in flight over one staging ring: Y = X C with X a part of
    the identity shows C itself."""
    n = 37 * 37
    A, g = Matrix(P.lap2d(37)[0]), np.random.default_rng(p)
    x = MultiVec(A, p, F64)
    x.set(np.asfortranarray(np.eye(n, p)))
    cs = [g.standard_normal((p, q)) for _ in range(4)]
    ys = [MultiVec(A, q, F64) for _ in cs]
    for c, y in zip(cs, ys):
        ops.lincomb(x, y, c)
    for c, y in zip(cs, ys):
        assert np.array_equal(y.get()[:p], c)
