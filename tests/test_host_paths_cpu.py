"""The library's host code -- which kernels a call launches, in which order,
what it keeps of the memory it takes, what it does where there is none --
against a HIP runtime of host memory (hostrt/hostrt.cpp), where no GPU is
needed.  Each test's script runs in a process of its own, because that runtime
has to be loaded before the library."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
rt.hostrt_launches.restype = C.c_char_p
rt.hostrt_live.restype = C.c_size_t
rt.hostrt_limit.argtypes = [C.c_size_t]
sys.path[:0] = sys.argv[2:]
import numpy as np
from gcge_hip import Matrix, MultiVec, Ops, capi
from gcge_hip import problems as P
F64, F32 = capi.GCGE_HIP_FP64, capi.GCGE_HIP_FP32
ops = Ops()
Hook = C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))

def launches(f):
    '''kernels that f() launches: [name, mangled template arguments and
    parameters, grid x, grid y]'''
    rt.hostrt_launches()
    f()
    out = []
    for line in rt.hostrt_launches().decode().splitlines():
        name, gx, gy = line.split()
        i = name.index("k_")
        j = i + int(name[:i].split("_1")[-1])
        out.append([name[i:j], name[j:], int(gx), int(gy)])
    return out

def launched(f):
    return [x[0] for x in launches(f)]
"""


@pytest.fixture(scope="session")
def hostrt(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hostrt") / "hostrt.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror",
                    os.path.join(HERE, "hostrt", "hostrt.cpp"), "-o", so], check=True)

    def run(script, **env):
        p = subprocess.run([sys.executable, "-c", PRELUDE + script, so, os.path.join(ROOT, "gcge-1.0_amd")],
                           capture_output=True, text=True, timeout=300, env={**os.environ, **env})
        assert p.returncode == 0, p.stdout + p.stderr

    return run


def test_columns_are_written_before_the_call_returns(hostrt):
    """A call that writes columns and returns sums of them reads the sums from
    a later launch, so the columns are complete, for every stream, when the
    host has the sums."""
    hostrt("""
A, M = P.lap3d_mass(8)
G = P.chung_lu(20000)[0]
for M, prec in ((P.lap2d(24)[0], F64), (P.lap2d(24)[0], F32), (M, F64), (G, F32)):
    A = Matrix(M)
    for k in (1, 2, 20):
        x, r, w, p = (MultiVec(A, k, prec) for _ in range(4))
        a = np.ones(k)
        for f in (lambda: ops.matdot_dot(A, x, w), lambda: ops.cg_update(x, 0, p, w, r, k, a),
                  lambda: ops.cg_residual_update(w, r, k, a), lambda: ops.pcg_residual_update(A, w, r, k, a)):
            names = launched(f)
            assert len(names) >= 2 and names[-1] == "k_reduce_rows_host", names
        assert launched(lambda: ops.dots(x, w))[0] == "k_dots"
""")


def test_host_columns_without_memory_for_the_row_order(hostrt):
    """Columns of an ordered matrix move and gradients map their entries on the
    host where the device has no room for the order, without an error."""
    hostrt("""
M = P.lap2d(300)[0]
n, k, g = M.shape[0], 4, np.random.default_rng(0)
X = np.asfortranarray(g.standard_normal((n, k)))
order = g.permutation(n).astype(np.int32)
plain, ordered = Matrix(M), Matrix(M, order=order)
stage = MultiVec(plain, k, F32)
stage.set(X)  # the staging buffer is there
jrp = np.arange(n + 1, dtype=np.int32)
jnz = g.integers(0, M.nnz, n).astype(np.int32)
jval, w, grad = g.standard_normal(n), np.ones(k), np.zeros(n)
px = MultiVec(plain, k, F64)

def gradient(A, mv):
    capi.load().GCGE_HIP_EigGradient(A.ptr, mv.ptr, k, w.ctypes.data_as(capi.DP), n, jrp.ctypes.data_as(capi.IP),
                                     jnz.ctypes.data_as(capi.IP), jval.ctypes.data_as(capi.DP),
                                     grad.ctypes.data_as(capi.DP))
    capi.raise_on_error("gradient")

entries = []

def note(name, args):
    if b"k_csr_gather_sum" in name:
        at = lambda i: C.c_void_p.from_address(args[i]).value
        e = np.ctypeslib.as_array((C.c_int * n).from_address(at(2))).copy()
        if at(4):
            e = np.ctypeslib.as_array((C.c_int * M.nnz).from_address(at(4)))[e]
        entries.append(e)

hook = Hook(note)
rt.hostrt_hook(hook)
gradient(plain, px)
room = MultiVec(ordered, k, F64)
gradient(ordered, room)
room.close()
fresh = Matrix(M, order=order)  # no order on the device yet
d, f = MultiVec(fresh, k, F64), MultiVec(fresh, k, F32)
rt.hostrt_limit(rt.hostrt_live())
for mv in (d, f):
    mv.set(X)
    assert np.array_equal(mv.get(), X if mv is d else X.astype(np.float32).astype(np.float64))
rt.hostrt_limit(rt.hostrt_live() + 4 * M.nnz)  # the rows of the entries, and no more
gradient(fresh, d)
assert np.array_equal(entries[0], jnz) and np.array_equal(entries[2], entries[1])
jnz[7] = M.nnz
try:
    gradient(fresh, d)
    raise SystemExit("a bad entry was taken")
except RuntimeError as e:
    assert "jnz[7]" in str(e), e
""")


def test_memory_of_gradients_and_host_columns_is_given_back(hostrt):
    """A large gradient keeps no more than 128 MiB and the entry order; what is
    kept makes room for an allocation that needs it, and goes with the last
    matrix."""
    hostrt("""
M = P.lap2d(300)[0]
n, k, g = M.shape[0], 3, np.random.default_rng(0)
plain, ordered = Matrix(M), Matrix(M, order=g.permutation(n).astype(np.int32))
x, y = MultiVec(ordered, k, F64), MultiVec(plain, k, F64)
X = np.asfortranarray(g.standard_normal((n, k)))
y.set(X)
ops.gram(y, y)  # scratch and coefficient staging are there
ops.lincomb(y, MultiVec(plain, 40, F64), np.ones((3, 40)))

def gradient(nj):
    jrp = np.linspace(0, nj, n + 1).astype(np.int32)
    jnz, jval = np.zeros(nj, np.int32), np.ones(nj)
    w, grad = np.ones(k), np.zeros(n)
    capi.load().GCGE_HIP_EigGradient(ordered.ptr, x.ptr, k, w.ctypes.data_as(capi.DP), n,
                                     jrp.ctypes.data_as(capi.IP), jnz.ctypes.data_as(capi.IP),
                                     jval.ctypes.data_as(capi.DP), grad.ctypes.data_as(capi.DP))
    capi.raise_on_error("gradient")

live = rt.hostrt_live()
held = capi.load().GCGE_HIP_DeviceBytes()
gradient(12_000_000)
fixed = 2 * 4 * M.nnz + 4 * n  # rows and order of the entries, row order
assert rt.hostrt_live() <= live + fixed, rt.hostrt_live() - live
gradient(5_000_000)
x.set(X)
x.get()
grown = rt.hostrt_live() - live
assert 0 < grown <= (128 << 20) + fixed
assert capi.load().GCGE_HIP_DeviceBytes() - held == grown
rt.hostrt_limit(rt.hostrt_live())
rows = 4 * M.nnz  # what no call gives back: the rows of the entries
cols = (grown - rows) // (8 * (n // 256 + 1 | 1) * 256)
big = MultiVec(plain, cols, F64)
big.close()
rt.hostrt_limit(1 << 40)
gradient(5_000_000)
for o in (x, y, ordered, plain):
    o.close()
assert rt.hostrt_live() < live, (rt.hostrt_live(), live)
assert rt.hostrt_live() <= 20 << 20, rt.hostrt_live()
""")


@pytest.mark.parametrize("layout,kernel", [("columns", "k_residual"), ("rows", "k_residual_rows"),
                                           ("halo", "k_residual_halo")])
def test_layout_override_holds_for_the_residual_check(hostrt, layout, kernel):
    """GCGE_HIP_SPMM_GATHER decides the residual check's kernel too, for rows of
    more than 8 entries on average in A, B or both."""
    hostrt(f"""
A, B = (Matrix(M) for M in P.lap3d_mass(12))
lam, idx = np.ones(5), np.arange(5, dtype=np.int32)
for prec in (F64, F32):
    x = MultiVec(A, 5, prec)
    for a, b in ((A, B), (B, None), (B, A), (B, B), (A, None)):
        names = launched(lambda: ops.residual_norms(a, b, x, idx, lam))
        assert "{kernel}" in names, (names, prec)
""", GCGE_HIP_SPMM_GATHER=layout)


def test_gather_kind_is_that_of_the_products(hostrt):
    """HIP_MatGatherKind names the kernel that products run with in the
    matrix's present precision: a grid's natural order may be staged in FP64 only."""
    hostrt("""
KERNELS = ["k_spmm", "k_spmm_rows", "k_spmm_halo"]
mats = [P.lap2d(40)[0], P.lap3d_mass(20)[1], P.chung_lu(20000)[0], P.lap3d_mass(85)[0]]
kinds = []
for M in mats:
    A = Matrix(M)
    kinds.append([])
    for prec in (F64, F32):
        A.set_precision(prec)
        kind = capi.load().HIP_MatGatherKind(A.ptr)
        kinds[-1].append(kind)
        A.set_precision(F64)
        x, y = MultiVec(A, 3, prec), MultiVec(A, 3, prec)
        assert KERNELS[kind] in launched(lambda: ops.matdot(A, x, y)), (kind, prec, A.n)
assert kinds == [[2, 2], [2, 2], [1, 1], [2, 0]], kinds
""")


def test_small_host_columns_are_ordered_and_converted_on_the_host(hostrt):
    """Where a launch, its wait and FP32's doubled bytes on the link cost more
    than the host's own work, no kernel runs; the columns are the same."""
    hostrt("""
M = P.lap2d(128)[0]
n, g = M.shape[0], np.random.default_rng(0)
plain, ordered = Matrix(M), Matrix(M, order=g.permutation(n).astype(np.int32))
# matrix, precision, columns, kernels of an upload and a download
UP, DOWN = ["k_rows_in"], ["k_rows_out"]
for A, prec, k, up, down in ((ordered, F64, 1, [], []), (ordered, F64, 2, [], []), (ordered, F64, 3, UP, DOWN),
                             (ordered, F32, 9, [], []), (ordered, F32, 10, UP, []), (ordered, F32, 20, UP, DOWN),
                             (plain, F32, 1, [], []), (plain, F32, 61, [], []), (plain, F32, 62, UP, []),
                             (plain, F32, 366, UP, []), (plain, F32, 367, UP, DOWN), (plain, F64, 100, [], [])):
    x = MultiVec(A, k, prec)
    X = np.asfortranarray(g.standard_normal((n, k)))
    assert launched(lambda: x.set(X)) == up, (prec, k)
    got = []
    assert launched(lambda: got.append(x.get())) == down, (prec, k)
    if not up and not down:
        assert np.array_equal(got[0], X if prec == F64 else X.astype(np.float32).astype(np.float64))
""")


def test_cut_of_the_slab_gram_kernel(tmp_path):
    """Every block's tiles fit its wavefronts, and the choice is cheap for many
    columns too."""
    exe = str(tmp_path / "gram_shape")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gcge-1.0_amd", "csrc"),
                    os.path.join(HERE, "hostrt", "gram_shape.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout


def test_matrix_without_host_memory_for_staged_blocks(hostrt):
    """A matrix whose staged blocks do not fit host memory takes another layout;
    nothing is thrown through the C entry."""
    hostrt("""
import resource
M = P.lap3d_mass(90)[1]
rowptr, col, val = M.indptr.astype(np.int32), M.indices.astype(np.int32), np.ascontiguousarray(M.data)
L = capi.load()
small = Matrix(P.lap3d_mass(12)[1])
with open("/proc/self/statm") as f:
    now = int(f.read().split()[0]) * resource.getpagesize()
device = 12 * M.nnz + 4 * M.shape[0]
resource.setrlimit(resource.RLIMIT_AS, (now + device + 24 * 1024 * 1024,) * 2)
A = L.HIP_MatCreateFromCSR(M.shape[0], M.shape[0], M.nnz, rowptr.ctypes.data_as(capi.IP),
                           col.ctypes.data_as(capi.IP), val.ctypes.data_as(capi.DP))
capi.raise_on_error("create")
assert L.HIP_MatGatherKind(A) == 1, L.HIP_MatGatherKind(A)
assert L.HIP_MatGatherKind(small.ptr) == 2
""")


def test_cleared_error_does_not_come_back(hostrt):
    """An allocation that failed is no error of the launches after
    GCGE_HIP_ClearError."""
    hostrt("""
A = Matrix(P.lap2d(40)[0])
x, y = MultiVec(A, 3, F64), MultiVec(A, 3, F64)
rt.hostrt_limit(rt.hostrt_live())
try:
    MultiVec(A, 3, F64)
    raise SystemExit("no error")
except RuntimeError as e:
    assert "out of memory" in str(e), e
rt.hostrt_limit(1 << 40)
ops.copy(x, y)
ops.dots(x, y)
""")


def test_kernel_of_a_combination(hostrt):
    """Few columns into many take the kernel without LDS while the blocks fit the
    cache and the other one does not fill the chip."""
    hostrt("""
for side, prec, p, q, rows in ((128, F64, 3, 200, 1), (128, F64, 12, 48, 0), (255, F64, 3, 300, 1), (255, F64, 20, 64, 1),
                               (255, F64, 48, 65, 0), (257, F64, 3, 300, 0), (128, F64, 64, 32, 1), (128, F64, 65, 32, 0),
                               (333, F32, 3, 200, 1), (333, F32, 20, 120, 1), (333, F32, 64, 65, 0),
                               (200, F32, 99, 65, 1), (200, F32, 128, 64, 1), (200, F32, 129, 64, 0),
                               (200, F32, 127, 33, 1), (200, F32, 128, 33, 0), (512, F32, 3, 65, 0),
                               (512, F32, 3, 64, 1), (800, F32, 12, 128, 0)):
    A = Matrix(P.lap2d(side)[0])
    x, y = MultiVec(A, p, prec), MultiVec(A, q, prec)
    names = launched(lambda: ops.lincomb(x, y, np.ones((p, q))))
    assert names[-1] == ("k_lincomb_rows" if rows else "k_lincomb_mfma"), (side, prec, p, q, names)
    for o in (x, y, A):
        o.close()
""")


def test_columns_of_a_search_update_meet_on_one_xcd(hostrt):
    """Workgroups go to the 8 XCDs in turn: with a multiple of 8 per column the
    same rows of every column, and the diagonal's, lie in one XCD's L2."""
    hostrt("""
for side in (3, 37, 300, 512, 1015):
    A = Matrix(P.lap2d(side)[0])
    for prec in (F64, F32):
        x, p, r = (MultiVec(A, 3, prec) for _ in range(3))
        (name, _, gx, gy), = [k for k in launches(lambda: ops.pcg_search_update(A, x, 0, p, r, 3, 3, np.ones(3),
                                                                                np.ones(3))) if "search" in k[0]]
        rows = 256 * (2 if prec == F64 else 4)
        assert gx % 8 == 0 and gy == 3 and gx * rows >= side * side, (side, prec, gx, gy)
        for o in (x, p, r):
            o.close()
    A.close()
""")


def test_accesses_of_the_element_wise_kernels(hostrt):
    """Copies store 16 bytes per thread in either direction of a conversion; the
    caches are passed by where the columns, each counted once, exceed 384 MB."""
    hostrt("""
A = Matrix(P.lap2d(40)[0])
v = {(p, i): MultiVec(A, 3, p) for p in (F64, F32) for i in (0, 1)}
for a, b, types in ((F64, F64, "IddLi2E"), (F64, F32, "IdfLi4E"), (F32, F64, "IfdLi2E"), (F32, F32, "IffLi4E")):
    (name, rest, _, _), = launches(lambda: ops.copy(v[a, 0], v[b, 1]))
    assert name == "k_copy" and rest.startswith(types), (name, rest)

B = Matrix(P.lap2d(1015)[0])
x, y = MultiVec(B, 24, F64), MultiVec(B, 24, F64)
for a, b, k, past in ((0.5, 0.5, 16, 0), (0.0, 0.5, 24, 0), (0.5, 0.5, 23, 0), (0.5, 0.5, 24, 1), (1.0, 0.0, 24, 1)):
    (name, rest, _, _), = launches(lambda: ops.axpby(a, x, b, y, k=k))
    assert name == "k_axpby" and rest.startswith("IdLi2ELb%dE" % past), (a, b, k, rest)
""")
