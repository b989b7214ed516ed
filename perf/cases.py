"""Timed cases of the GCGE backend: what an eigenvalue computation has it do.

A case is a dict of plain values.  ``kind`` says which calls one pass makes,
all of them through ``gcge_hip``:

* ``pcg``       a block CG solve of A X = B for k right-hand sides with a
                fixed number of steps (SpMM with fused dots, residual update,
                search update), Jacobi-preconditioned or plain: the inner
                solves that build the W block, where a solve spends most of
                its time;
* ``rr``        one Rayleigh-Ritz update: A W, V^T (A W) and X = V C;
* ``orth``      W against V and itself: projection, CholQR factor, W R^-1,
                with or without a mass matrix;
* ``spmm``      one product A X (with dots x_j . y_j when ``dot``);
* ``residual``  the convergence check: norms of A x - lambda B x, x and B x;
* ``gradient``  d(sum w_i lambda_i)/d theta (the backward direction), from
                host eigenvectors as the call takes them;
* ``solve``     a whole eigensolve from a given block.

Operators are the generators of ``gcge_hip.problems`` by name and grid size
``m`` (``chung_lu``: vertices).  ``order`` "tiles" lists a grid's rows in
8 x 8 x 8 (16 x 16 in 2-D) tiles, as ``HIP_MatLocalityOrder`` does;
"natural" is the caller's own order.  Multivectors are returned as they lie
in HBM (one row per column of the block, rows in the matrix's order).
"""
from __future__ import annotations

import ctypes
import functools
import itertools
import math
import os
import sys
import types

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gcge-1.0_amd"))
# torch brings GNU OpenMP into the process; the host MKL that the subspace
# problems call has to use the same runtime
os.environ.setdefault("MKL_THREADING_LAYER", "GNU")

import gcge_hip as G  # noqa: E402
from gcge_hip import capi, problems as P  # noqa: E402

PREC = {"f64": capi.GCGE_HIP_FP64, "f32": capi.GCGE_HIP_FP32}
DTYPE = {"f64": torch.float64, "f32": torch.float32}
SIZE = {"f64": 8, "f32": 4}


# --------------------------------------------------------------- the cases

def listed():
    return [
        # the 128 x 128 Laplacian with 20 vectors: one block fits a cache, so
        # launches and the host's reads of the dots decide
        dict(name="pcg lap2d small", kind="pcg", op="lap2d", m=128, order="tiles", k=20, dtype="f64", precond=False,
             steps=20),
        # the FP32 inner solves of the mixed path at the benchmark's size,
        # with the number of columns that are active on average
        dict(name="pcg 3d f32", kind="pcg", op="vardiff3d", m=160, order="tiles", k=48, dtype="f32", precond=True,
             steps=6),
        # the FP64 inner solves with the same settings, an odd column count
        dict(name="pcg 3d f64", kind="pcg", op="vardiff3d", m=144, order="tiles", k=33, dtype="f64", precond=True,
             steps=4),
        # the drop-in default: the caller's row order, plain CG, an odd grid
        dict(name="pcg 3d natural", kind="pcg", op="vardiff3d", m=101, order="natural", k=35, dtype="f64",
             precond=False, steps=4),
        # Rayleigh-Ritz over [X P W] with 100 columns each, benchmark size
        dict(name="rr 3d f64", kind="rr", op="vardiff3d", m=160, order="tiles", p=300, k=100, dtype="f64"),
        # W orthonormalization of the FP32 phase, B = I
        dict(name="orth 3d f32", kind="orth", op="vardiff3d", m=128, order="tiles", p=200, k=100, dtype="f32"),
        # the same for a generalized problem: 27-point mass matrix, FP64
        dict(name="orth mass f64", kind="orth", op="lap3d_mass", m=96, order="tiles", p=100, k=50, dtype="f64"),
        # a random graph with a power-law degree distribution
        dict(name="spmm graph f32", kind="spmm", op="chung_lu", m=1_000_000, order="natural", k=64, dtype="f32",
             dot=True),
        # the convergence check of 100 pairs, B = I and B = mass
        dict(name="residual 3d f64", kind="residual", op="vardiff3d", m=160, order="tiles", k=100, dtype="f64"),
        dict(name="residual mass f64", kind="residual", op="lap3d_mass", m=96, order="tiles", k=50, dtype="f64"),
        # gradient of the 16 lowest eigenvalues on the 512 x 512 grid
        dict(name="gradient 2d", kind="gradient", op="vardiff2d", m=512, order="natural", k=16, dtype="f64"),
        # whole solves with the mixed path: the generalized 3-D problem
        dict(name="solve mass mixed", kind="solve", op="lap3d_mass", m=64, order="tiles", nev=50, precision="mixed"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["pcg", "rr", "orth", "spmm", "residual", "gradient", "solve"], [7, 2, 3, 2, 3, 1, 2])[0]
    if kind == "solve":
        op = rng.choice(["lap2d", "vardiff2d", "lap3d_mass", "vardiff3d"])
        hi = {"lap2d": 200, "vardiff2d": 256, "lap3d_mass": 48, "vardiff3d": 64}[op]
        return dict(kind="solve", op=op, m=_log(rng, hi // 4 + 4, hi), order="tiles", nev=_log(rng, 6, 40),
                    precision="mixed")
    if kind == "gradient":
        return dict(kind="gradient", op="vardiff2d", m=_log(rng, 48, 512), order=rng.choice(["natural", "tiles"]),
                    k=_log(rng, 1, 32), dtype="f64")
    ops = ["lap2d", "vardiff2d", "vardiff3d"]
    if kind in ("orth", "residual", "spmm"):
        ops += ["lap3d_mass"] * 2
    if kind in ("spmm", "residual"):
        ops += ["chung_lu"]
    op = rng.choice(ops)
    lo, hi = {"lap2d": (64, 1024), "vardiff2d": (64, 1024), "vardiff3d": (20, 144), "lap3d_mass": (20, 96),
              "chung_lu": (20_000, 1_000_000)}[op]
    c = dict(kind=kind, op=op, m=_log(rng, lo, hi),
             order="natural" if op == "chung_lu" else rng.choice(["tiles", "tiles", "natural"]))
    c["dtype"] = rng.choice(["f64", "f32"])
    if kind == "pcg":
        c.update(k=_log(rng, 1, 64), precond=rng.random() < 0.6, steps=rng.randint(2, 6))
    elif kind in ("rr", "orth"):
        k = _log(rng, 2, 100)
        c.update(p=k * rng.randint(1, 3) + rng.randint(0, 7), k=k)
        if kind == "rr" and rng.random() < 0.7:
            c["dtype"] = "f64"
    elif kind == "spmm":
        c.update(k=_log(rng, 1, 100), dot=rng.random() < 0.5)
    else:
        c.update(k=_log(rng, 1, 100))
    return c


# --------------------------------------------------------------- operators

class Csr(types.SimpleNamespace):
    """What gcge_hip.Matrix reads of a CSR matrix (shape, indptr, indices,
    data), and the same entries padded to a rectangle (cols, vals)."""


def _grid(shape, offsets):
    """CSR of a grid operator: ``offsets`` maps an offset tuple to the value
    at every cell (array of ``shape`` or a number); entries that leave the
    grid are dropped, columns ascend within a row."""
    n = int(np.prod(shape))
    idx = np.indices(shape, dtype=np.int32, sparse=True)
    stride = [int(np.prod(shape[a + 1:])) for a in range(len(shape))]
    items = sorted(offsets.items(), key=lambda it: sum(o * s for o, s in zip(it[0], stride)))
    cols = np.empty((n, len(items)), np.int32)
    vals = np.empty((n, len(items)))
    keep = np.empty((n, len(items)), bool)
    row = np.arange(n, dtype=np.int32)
    for e, (off, v) in enumerate(items):
        ok = np.ones(shape, bool)
        for a, o in enumerate(off):
            ok &= (idx[a] + o >= 0) & (idx[a] + o < shape[a])
        ok = ok.ravel()
        keep[:, e] = ok
        cols[:, e] = np.where(ok, row + sum(o * s for o, s in zip(off, stride)), row)
        vals[:, e] = np.where(ok, np.broadcast_to(v, shape).ravel(), 0.0)
    indptr = np.zeros(n + 1, np.int32)
    np.cumsum(keep.sum(axis=1), out=indptr[1:])
    return Csr(shape=(n, n), indptr=indptr, indices=cols[keep], data=vals[keep], nnz=int(indptr[-1]), cols=cols,
               vals=vals)


def _laplace(d, m):
    off = {(0,) * d: 2.0 * d}
    for a in range(d):
        for o in (-1, 1):
            off[tuple(o if b == a else 0 for b in range(d))] = -1.0
    return _grid((m,) * d, off)


def _diffusion(kappa, scale):
    """Finite volumes with harmonic-mean faces and Dirichlet walls, the
    operator of problems.fv_diffusion."""
    shape, d = kappa.shape, kappa.ndim
    off, diag = {}, np.zeros(shape)
    for a in range(d):
        k1 = np.moveaxis(kappa, a, 0)
        t = scale[a] * 2.0 * k1[:-1] * k1[1:] / (k1[:-1] + k1[1:])
        for o in (-1, 1):
            v = np.zeros(shape)
            w, g = np.moveaxis(v, a, 0), np.moveaxis(diag, a, 0)
            (w[1:] if o < 0 else w[:-1])[...] = -t
            (g[1:] if o < 0 else g[:-1])[...] += t
            g[0 if o < 0 else -1] += scale[a] * 2.0 * k1[0 if o < 0 else -1]
            off[tuple(o if b == a else 0 for b in range(d))] = v
    off[(0,) * d] = diag
    return _grid(shape, off)


@functools.lru_cache(maxsize=2)
def _host(op, m):
    """(A, B or None) on the host."""
    if op == "lap2d":
        return _laplace(2, m), None
    if op == "vardiff2d":
        return _diffusion(P.vardiff2d_theta(m), (1.0, 1.3)), None
    if op == "vardiff3d":
        return _diffusion(np.exp(P.gaussian_field((m, m, m), 8.0, 1.0, 0)), (1.0, 1.0, 1.0)), None
    if op == "lap3d_mass":
        h = 1.0 / (m + 1)
        mass = {o: h ** 3 / 216.0 * math.prod((1.0, 4.0, 1.0)[i + 1] for i in o)
                for o in itertools.product((-1, 0, 1), repeat=3)}
        return _laplace(3, m), _grid((m, m, m), mass)
    if op == "chung_lu":
        M = P.chung_lu(m)[0]
        return M, None
    raise ValueError(op)


def _dim(op):
    return 3 if op in ("vardiff3d", "lap3d_mass") else 2


@functools.lru_cache(maxsize=2)
def _tiles(op, m):
    """perm[new position] = row: tile by tile, both levels lexicographic."""
    t = 8 if _dim(op) == 3 else 16
    c = np.indices((m,) * _dim(op), dtype=np.int64).reshape(_dim(op), -1)
    key = np.zeros(c.shape[1], np.int64)
    for part in (c // t, c % t):
        for a in part:
            key = key * (m // t + t + 1) + a
    return np.argsort(key, kind="stable").astype(np.int32)


@functools.lru_cache(maxsize=3)
def _device(op, m, order):
    """The matrices a program uploads once: (A, B or None)."""
    A, B = _host(op, m)
    perm = _tiles(op, m) if order == "tiles" else None
    return G.Matrix(A, order=perm), None if B is None else G.Matrix(B, order=perm)


# --------------------------------------------------------------- inputs

class _Handle(ctypes.Structure):
    """Head of a multivector handle's struct."""
    _fields_ = [("magic", ctypes.c_uint32), ("prec", ctypes.c_int), ("n", ctypes.c_int64), ("ld", ctypes.c_int64),
                ("ncols", ctypes.c_int), ("data", ctypes.c_void_p)]


def _view(mv):
    """The multivector's columns in HBM as an (ncols, n) tensor, no copy;
    the tensor keeps the multivector alive."""
    h = _Handle.from_address(mv.ptr)
    w = 8 if h.prec == capi.GCGE_HIP_FP64 else 4
    iface = dict(shape=(h.ncols, h.n), strides=(h.ld * w, w), typestr="<f%d" % w, data=(h.data, False), version=3)
    t = torch.as_tensor(types.SimpleNamespace(__cuda_array_interface__=iface, owner=mv), device="cuda")
    t.owner = mv
    return t


def _blocks(seed, tag, k, n, dtype):
    """k columns of normal values, 16 at a time (from the seed alone)."""
    g = torch.Generator("cuda").manual_seed(1_000_003 * int(seed) + tag)
    for c in range(0, k, 16):
        yield c, torch.randn(min(16, k - c), n, generator=g, device="cuda", dtype=DTYPE[dtype])


def _random(seed, tag, k, n, dtype, scale=1.0):
    return torch.cat([b for _, b in _blocks(seed, tag, k, n, dtype)]) * scale


def _filled(mat, k, dtype, seed=None, tag=0, scale=1.0):
    """A new multivector of k columns, filled from the seed when given."""
    mv = G.MultiVec(mat, k, PREC[dtype])
    G.synchronize()
    if seed is not None:
        v = _view(mv)
        for c, b in _blocks(seed, tag, k, mat.n, dtype):
            v[c:c + b.shape[0]] = b * scale
        torch.cuda.synchronize()
    return mv


def _coef(seed, p, q):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal((p, q)) / math.sqrt(p))


def _vscale(case, n):
    """Scale of random columns whose B-norm is then about 1."""
    return (n * (64.0 / 216.0 / (case["m"] + 1) ** 3 if case["op"] == "lap3d_mass" else 1.0)) ** -0.5


@functools.lru_cache(maxsize=2)
def _jacobian(m):
    """Jacobian of the stored values of vardiff2d(m) by its cells."""
    A, _ = _host("vardiff2d", m)
    return P.fv_diffusion_jacobian(P.vardiff2d_theta(m), A, (1.0, 1.3))


def _pairs(case, seed, n):
    r = np.random.default_rng(seed)
    X = np.asfortranarray(r.standard_normal((case["k"], n)).T / math.sqrt(n))
    return X, r.uniform(0.5, 2.0, case["k"])


@functools.lru_cache(maxsize=1)
def _ops():
    return G.Ops()


def prepare(case, seed):
    A, B = _device(case["op"], case["m"], case["order"])
    s = types.SimpleNamespace(case=case, ops=_ops(), A=A, B=B)
    n, kind, dt, k = A.n, case["kind"], case.get("dtype"), case.get("k")
    if kind == "pcg":
        s.b = _filled(A, k, dt, seed)
        s.x, s.r, s.p, s.w = (_filled(A, k, dt) for _ in range(4))
        s.out = [_view(v) for v in (s.x, s.r, s.p)]
    elif kind == "rr":
        s.V = _filled(A, case["p"], dt, seed, 0, n ** -0.5)
        s.T, s.X = _filled(A, k, dt), _filled(A, k, dt)
        s.C = _coef(seed, case["p"], k)
        s.out = [_view(s.T), _view(s.X)]
    elif kind == "orth":
        s.V = _filled(A, case["p"], dt, seed, 0, _vscale(case, n))
        s.W0 = _filled(A, k, dt, seed, 1, _vscale(case, n))
        s.W, s.T, s.Q = (_filled(A, k, dt) for _ in range(3))
        s.out = [_view(s.W), _view(s.Q)]
    elif kind == "spmm":
        s.x, s.y = _filled(A, k, dt, seed), _filled(A, k, dt)
        s.M = B if B is not None else A
        s.out = [_view(s.y)]
    elif kind == "residual":
        s.x = _filled(A, k, dt, seed)
        s.lam = np.random.default_rng(seed).uniform(0.1, 4.0, k)
        s.idx = np.arange(k, dtype=np.int32)
    elif kind == "gradient":
        s.X, s.wgt = _pairs(case, seed, n)
        s.J = _jacobian(case["m"])
    else:
        s.X0 = _filled(A, case["nev"], "f64", seed)
        s.solver = G.Solver(A, B, case["nev"], precision=case["precision"], opt_rr_eig_partly=1, conv_type="NS",
                            ev_tol=1e-8, ev_max_it=2000)
    G.synchronize()
    return s


# --------------------------------------------------------------- one pass

def _pcg(s):
    c, o = s.case, s.ops
    k, zero = c["k"], np.zeros(c["k"])
    o.copy(s.b, s.r)
    o.axpby(0.0, s.x, 0.0, s.x)
    if c["precond"]:
        rho, rr = o.pcg_residual_update(s.A, s.w, s.r, k, zero)
        o.pcg_search_update(s.A, s.x, 0, s.p, s.r, 0, k, zero, zero)
    else:
        rho = rr = o.dots(s.r, s.r)
        o.axpby(1.0, s.r, 0.0, s.p)
    for _ in range(c["steps"]):
        alpha = rho / o.matdot_dot(s.A, s.p, s.w)
        last = rho
        if c["precond"]:
            rho, rr = o.pcg_residual_update(s.A, s.w, s.r, k, alpha)
            o.pcg_search_update(s.A, s.x, 0, s.p, s.r, k, k, alpha, rho / last)
        else:
            rho = rr = o.cg_residual_update(s.w, s.r, k, alpha)
            o.cg_search_update(s.x, 0, s.p, s.r, k, k, alpha, rho / last)
    return s.out + [rr]


def _orth(s):
    o = s.ops

    def bw():
        if s.B is None:
            return s.W
        o.matdot(s.B, s.W, s.T)
        return s.T

    o.copy(s.W0, s.W)
    g = o.gram(s.V, bw())
    o.lincomb(s.V, s.W, g, alpha=-1.0, beta=1.0)
    sw = o.gram(s.W, bw(), sym=True)
    o.lincomb(s.W, s.Q, np.linalg.inv(np.linalg.cholesky(sw)).T)
    return s.out + [g, sw]


def run(s):
    kind, o = s.case["kind"], s.ops
    if kind == "pcg":
        return _pcg(s)
    if kind == "rr":
        k, p = s.case["k"], s.case["p"]
        o.matdot(s.A, s.V, s.T, xs=p - k, k=k)
        g = o.gram(s.V, s.T)
        o.lincomb(s.V, s.X, s.C)
        return s.out + [g]
    if kind == "orth":
        return _orth(s)
    if kind == "spmm":
        if s.case["dot"]:
            return s.out + [o.matdot_dot(s.M, s.x, s.y)]
        o.matdot(s.M, s.x, s.y)
        return s.out
    if kind == "residual":
        return list(o.residual_norms(s.A, s.B, s.x, s.idx, s.lam))
    if kind == "gradient":
        return G.eig_gradient(s.A, s.X, s.wgt, s.A.n, *s.J)
    # the eigenvectors are fixed only up to the tolerance and, in a cluster,
    # up to a rotation; the eigenvalues are what two solves share
    r = s.solver.solve(s.X0, keep_evec=False)
    return [r["eval"], r["rc"]]


# --------------------------------------------------------------- work

def work(case):
    """Bytes and operations of the calls of one pass: for each call its
    inputs read once and its outputs written once (whole solves: the same
    for a nominal course of 20 outer iterations with 20 inner steps)."""
    op, m = case["op"], case["m"]
    n = m if op == "chung_lu" else m ** _dim(op)
    row = {"lap2d": 5, "vardiff2d": 5, "vardiff3d": 7, "lap3d_mass": 7, "chung_lu": 17}[op]
    kind = case["kind"]
    w = SIZE[case.get("dtype", "f64")]
    k = case.get("k", 0)

    def spmm(per_row, cols, size):
        return n * (per_row * (size + 4) + 4 + 2 * cols * size), 2 * per_row * n * cols

    if kind == "pcg":
        b, f = spmm(row, k, w)
        d = n * w if case["precond"] else 0
        s = case["steps"]
        return dict(bytes=s * (b + 8 * n * k * w + 2 * d) + 5 * n * k * w, flops=s * (f + 10 * n * k))
    if kind == "rr":
        b, f = spmm(row, k, w)
        p = case["p"]
        return dict(bytes=b + 2 * n * (p + k) * w, flops=f + 4 * n * p * k)
    if kind == "orth":
        p = case["p"]
        b, f = spmm(27, k, w) if op == "lap3d_mass" else (0, 0)
        return dict(bytes=2 * b + n * w * (2 * (p + k) + 6 * k), flops=2 * f + 4 * n * p * k + 3 * n * k * k)
    if kind == "spmm":
        b, f = spmm(27 if op == "lap3d_mass" else row, k, w)
        return dict(bytes=b, flops=f)
    if kind == "residual":
        e = row + (27 if op == "lap3d_mass" else 0)
        return dict(bytes=n * (12 * e + 4 + k * w), flops=2 * n * e * k)
    if kind == "gradient":
        e = row * n
        return dict(bytes=n * k * 8 + e * 12 + 13 * n * 12 + 8 * n, flops=3 * e * k + 26 * n)
    nev = case["nev"]
    b, f = spmm(row, nev, 4)
    return dict(bytes=400 * (b + 8 * n * nev * 4) + 20 * n * 12 * nev * 8,
                flops=400 * (f + 10 * n * nev) + 20 * 16 * n * nev * nev)


# --------------------------------------------------------------- 64 bits

def _order(case, n):
    return _tiles(case["op"], case["m"]) if case["order"] == "tiles" else np.arange(n, dtype=np.int32)


def _apply(M, case):
    """X -> M X for rows of X in the case's order, X an (k, n) f64 tensor."""
    n = M.shape[0]
    if case["op"] == "chung_lu":
        return lambda X: torch.from_numpy(np.ascontiguousarray((M @ X.cpu().numpy().T).T)).cuda()
    perm = torch.from_numpy(_order(case, n).astype(np.int64)).cuda()
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(n, device="cuda")
    cols = [inv[torch.from_numpy(M.cols[:, e].astype(np.int64)).cuda()][perm] for e in range(M.cols.shape[1])]
    vals = [torch.from_numpy(M.vals[:, e].copy()).cuda()[perm] for e in range(M.cols.shape[1])]

    def times(X):
        Y = torch.zeros_like(X)
        for j in range(X.shape[0]):
            for c, v in zip(cols, vals):
                Y[j] += v * X[j][c]
        return Y

    return times


def _exact_pcg(case, seed, A, n):
    b = _random(seed, 0, case["k"], n, case["dtype"]).double()
    times = _apply(A, case)
    if case["precond"]:
        d = np.zeros(n)
        d[:] = np.where(A.cols == np.arange(n)[:, None], A.vals, 0.0).sum(axis=1)
        di = torch.from_numpy(1.0 / d[_order(case, n)]).cuda()
    else:
        di = torch.ones(n, device="cuda", dtype=torch.float64)
    x, r = torch.zeros_like(b), b
    p = r * di
    rho = (r * p).sum(1)
    for _ in range(case["steps"]):
        w = times(p)
        a = (rho / (p * w).sum(1))[:, None]
        x += a * p
        r = r - a * w
        z = r * di
        new = (r * z).sum(1)
        p = z + (new / rho)[:, None] * p
        rho = new
    return [x, r, p, (r * r).sum(1).cpu().numpy()]


def exact(case, seed):
    A, B = _host(case["op"], case["m"])
    n, kind = A.shape[0], case["kind"]
    if kind == "pcg":
        return _exact_pcg(case, seed, A, n)
    if kind == "rr":
        V = _random(seed, 0, case["p"], n, case["dtype"], n ** -0.5).double()
        T = _apply(A, case)(V[case["p"] - case["k"]:])
        C = torch.from_numpy(_coef(seed, case["p"], case["k"])).cuda()
        return [T, C.T @ V, (V @ T.T).cpu().numpy()]
    if kind == "orth":
        V = _random(seed, 0, case["p"], n, case["dtype"], _vscale(case, n)).double()
        W = _random(seed, 1, case["k"], n, case["dtype"], _vscale(case, n)).double()
        times = (lambda X: X) if B is None else _apply(B, case)
        g = V @ times(W).T
        W = W - g.T @ V
        sw = W @ times(W).T
        sw = torch.triu(sw) + torch.triu(sw, 1).T
        Q = torch.linalg.inv(torch.linalg.cholesky(sw)) @ W
        return [W, Q, g.cpu().numpy(), sw.cpu().numpy()]
    if kind == "spmm":
        X = _random(seed, 0, case["k"], n, case["dtype"]).double()
        Y = _apply(B if B is not None else A, case)(X)
        return [Y, (X * Y).sum(1).cpu().numpy()] if case["dot"] else [Y]
    if kind == "residual":
        X = _random(seed, 0, case["k"], n, case["dtype"]).double()
        lam = torch.from_numpy(np.random.default_rng(seed).uniform(0.1, 4.0, case["k"])).cuda()
        BX = X if B is None else _apply(B, case)(X)
        R = _apply(A, case)(X) - lam[:, None] * BX
        return [torch.linalg.vector_norm(v, dim=1).cpu().numpy() for v in (R, X, BX)]
    if kind == "gradient":
        X, wgt = _pairs(case, seed, n)
        rows = np.repeat(np.arange(n), np.diff(A.indptr))
        g = sum(wgt[i] * X[rows, i] * X[A.indices, i] for i in range(case["k"]))
        jp, jn, jv = _jacobian(case["m"])
        return np.add.reduceat(np.append(jv * g[jn], 0.0), jp[:-1])
    # eigenvalues: closed forms where the grid has them
    return [_closed(case), None] if case["op"] in ("lap2d", "lap3d_mass") else None


def _closed(case):
    """Lowest eigenvalues of the constant-coefficient grids."""
    m, nev = case["m"], case["nev"]
    t = np.arange(1, m + 1) * math.pi / (m + 1)
    a = 2.0 - 2.0 * np.cos(t)
    if case["op"] == "lap2d":
        return np.sort((a[:, None] + a[None, :]).ravel())[:nev]
    mu = (4.0 + 2.0 * np.cos(t)) / (6.0 * (m + 1))
    lam = (a[:, None, None] + a[None, :, None] + a[None, None, :]) / (
        mu[:, None, None] * mu[None, :, None] * mu[None, None, :])
    return np.sort(lam.ravel())[:nev]
