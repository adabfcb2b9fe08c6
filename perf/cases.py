"""Workloads of the Krylov-Schur framework through its public entry points, for
timing and for comparing results.

A case is a plain dict.  ``listed()`` gives the fixed ones, ``draw(rng)`` one more
from the same ranges, ``prepare(case, seed)`` what a program holds before the call
(matrices on the device, bases, solver objects), ``run(state)`` one pass,
``work(case)`` the bytes and operations the pass cannot do without,
``tolerance(case)`` the differences another correct implementation would show and
``exact(case, seed)`` the same results from plain torch in 64 bits.

Kinds:

* ``solve``    a whole EPSSolve with its eigenvectors (standard, mixed precision, two-sided)
* ``serve``    a burst of requests through the serving loop
* ``expand``   BVMatArnoldi: some columns added to a Krylov basis
* ``spmv``     one product with a CSR matrix
* ``block``    BVOrthogonalize of a block of columns
* ``lu``       the direct shift-and-invert: factorization and a few solves
* ``inner``    one iterative inner solve of shift-and-invert
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from slepc_amd import eps as E
from slepc_amd import ks
from slepc_amd import matgen as M
from slepc_amd import serve as S

DEV = "cuda"
BLOCKS = {"gs": E.BV.GS, "chol": E.BV.CHOL, "tsqr": E.BV.TSQR, "tsqrchol": E.BV.TSQRCHOL}


def listed():
    return [
        # a small graph Laplacian, the common request of a serving front end solved alone: launches count
        {"name": "solve-er-2000", "kind": "solve", "matrix": "er", "size": 2000, "nev": 8, "ncv": 32, "mixed": 0.0,
         "twosided": False},
        # the benchmark's problem: variable-coefficient Laplacian 128^3, the largest whole solve
        {"name": "solve-varcoef-128", "kind": "solve", "matrix": "varcoef", "size": 128, "nev": 16, "ncv": 48,
         "mixed": 0.0, "twosided": False},
        # right and left eigenvectors of a nonsymmetric operator
        {"name": "twosided-convdiff-150", "kind": "solve", "matrix": "convdiff", "size": 150, "nev": 4, "ncv": 24,
         "mixed": 0.0, "twosided": True},
        # a burst of graph requests of mixed sizes, eight at a time on the device
        {"name": "serve-er-16", "kind": "serve", "requests": 16, "nmax": 100000},
        # the FP32 phase of the mixed form: the last columns before a restart on a 2048^2 operator
        {"name": "expand-f32-convdiff-2048", "kind": "expand", "matrix": "convdiff", "size": 2048, "k": 32, "steps": 8,
         "prec": "f32"},
        # a wide basis (large nev): columns beyond 128 of an odd-sized problem
        {"name": "expand-f64-varcoef-74-wide", "kind": "expand", "matrix": "varcoef", "size": 74, "k": 192, "steps": 8,
         "prec": "f64"},
        # power-law graph with FP32 values and FP64 vectors: irregular rows, hub rows, scattered gathers
        {"name": "spmv-rmat-20", "kind": "spmv", "matrix": "rmat", "size": 20, "vprec": "f32", "xprec": "f64"},
        # block orthogonalization: Gram matrix, Cholesky, X R^-1
        {"name": "chol-1000003x48", "kind": "block", "n": 1000003, "k": 48, "block": "chol"},
        # block orthogonalization where Cholesky is not safe: TSQR with explicit Q
        {"name": "tsqr-500000x32", "kind": "block", "n": 500000, "k": 32, "block": "tsqr"},
        # shift-and-invert with the default direct solver: factorization and four solves
        {"name": "lu-128x127", "kind": "lu", "nx": 128, "ny": 127, "solves": 4},
        # shift-and-invert with an inner CG: one application of the operator
        {"name": "cg-256x255", "kind": "inner", "method": "cg", "nx": 256, "ny": 255, "peclet": 0.0},
        # a nonsymmetric operator: BiCGStab with ILU(0), one application
        {"name": "bcgs-ilu-128x127", "kind": "inner", "method": "bcgs-ilu", "nx": 128, "ny": 127, "peclet": 5.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "serve", "expand", "expand", "spmv", "block", "block", "lu", "inner"])
    if kind == "solve":
        matrix = rng.choice(["er", "varcoef", "convdiff"])
        size = {"er": _log(rng, 1000, 200000), "varcoef": _log(rng, 12, 120), "convdiff": _log(rng, 40, 700)}[matrix]
        nev = rng.randint(4, 16)
        mixed = 1e-5 if matrix == "convdiff" and rng.random() < 0.4 else 0.0
        two = matrix == "convdiff" and mixed == 0.0 and rng.random() < 0.6
        if two:
            size, nev = min(size, 300), min(nev, 6)
        return {"kind": "solve", "matrix": matrix, "size": size, "nev": nev, "ncv": 2 * nev + 16, "mixed": mixed,
                "twosided": two}
    if kind == "serve":
        return {"kind": "serve", "requests": rng.randint(3, 16), "nmax": _log(rng, 4000, 100000)}
    if kind == "expand":
        matrix = rng.choice(["varcoef", "convdiff"])
        size = _log(rng, 12, 128) if matrix == "varcoef" else _log(rng, 40, 2048)
        n = size ** 3 if matrix == "varcoef" else size ** 2
        prec = rng.choice(["f64", "f64", "f32"])
        k = min(_log(rng, 4, 248), n // 4, max(4, int(1.2e8 // n)))
        return {"kind": "expand", "matrix": matrix, "size": size, "k": k, "steps": rng.randint(4, 12), "prec": prec}
    if kind == "spmv":
        matrix = rng.choice(["rmat", "er", "varcoef", "grid"])
        size = {"rmat": rng.randint(14, 20), "er": _log(rng, 20000, 400000), "varcoef": _log(rng, 40, 128),
                "grid": _log(rng, 320, 2048)}[matrix]
        vprec = "f32" if matrix == "rmat" else rng.choice(["f64", "f64", "f32"])
        return {"kind": "spmv", "matrix": matrix, "size": size, "vprec": vprec,
                "xprec": rng.choice(["f64", "f32"]) if vprec == "f32" else "f64"}
    if kind == "block":
        block = rng.choice(["chol", "chol", "tsqr", "tsqr", "tsqrchol", "gs"])
        k = _log(rng, 3, 60)
        return {"kind": "block", "n": _log(rng, 1000, min(1500000, int(4.8e7 // k))), "k": k, "block": block}
    if kind == "lu":
        nx = _log(rng, 12, 126)
        return {"kind": "lu", "nx": nx, "ny": max(5, nx - rng.randint(1, 5)), "solves": rng.randint(1, 6)}
    method = rng.choice(["cg", "cg", "bcgs", "bcgs-ilu"])
    nx = _log(rng, 16, {"cg": 512, "bcgs": 256, "bcgs-ilu": 140}[method])
    return {"kind": "inner", "method": method, "nx": nx, "ny": max(5, nx - rng.randint(1, 5)),
            "peclet": 0.0 if method == "cg" else rng.uniform(1.0, 8.0)}


# ------------------------------------------------------------------ matrices and inputs
def _matrix(case, seed):
    """Host CSR (rowptr, colidx, val) of a case's operator."""
    size = case["size"]
    if case["matrix"] == "er":
        return M.er_laplacian(size, 8.0, seed=seed)
    if case["matrix"] == "varcoef":
        return M.varcoef_laplacian_3d(size, seed=seed)
    if case["matrix"] == "convdiff":
        return M.convection_diffusion_2d(size, seed=seed)
    if case["matrix"] == "rmat":
        return M.rmat_shifted_normalized_laplacian(size, seed=seed)
    return _grid(size, size - 3, 0.0)     # "grid": an odd 5-point operator


def _rows(case):
    size = case["size"]
    return {"er": size, "varcoef": size ** 3, "convdiff": size ** 2, "rmat": 2 ** min(size, 40),
            "grid": size * (size - 3)}[case["matrix"]]


def _nnz(case):
    """Stored entries, to a few per cent."""
    return int(_rows(case) * {"er": 9, "varcoef": 7, "convdiff": 5, "rmat": 31, "grid": 5}[case["matrix"]])


def _grid(nx, ny, peclet):
    """-u'' + peclet u' in both directions, central differences: constant coefficients, so the
    eigenvectors are scaled sines in each direction (see _grid_solve)."""
    n = nx * ny
    cx, cy = peclet / (2.0 * (nx + 1)), peclet / (2.0 * (ny + 1))
    i = np.arange(n, dtype=np.int64)
    x, y = i % nx, i // nx
    cols = np.stack([i - nx, i - 1, i, i + 1, i + nx], axis=1)
    vals = np.broadcast_to(np.array([-1.0 - cy, -1.0 - cx, 4.0, -1.0 + cx, -1.0 + cy]), cols.shape)
    keep = np.stack([y > 0, x > 0, np.ones(n, bool), x < nx - 1, y < ny - 1], axis=1)
    rowptr = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(keep.sum(axis=1), out=rowptr[1:])
    return rowptr.astype(np.int32), cols[keep].astype(np.int32), np.ascontiguousarray(vals[keep])


def _grid_axis(n, peclet):
    c = peclet / (2.0 * (n + 1))
    j = torch.arange(1, n + 1, dtype=torch.float64, device=DEV)
    s = torch.sin(torch.outer(j, j) * (math.pi / (n + 1))) * math.sqrt(2.0 / (n + 1))
    lam = 2.0 - 2.0 * math.sqrt(1.0 - c * c) * torch.cos(j * (math.pi / (n + 1)))
    d = ((1.0 + c) / (1.0 - c)) ** (j / 2.0)
    return s, lam, d


def _grid_solve(nx, ny, peclet, sigma, b):
    """(A - sigma I)^-1 b of _grid's operator by its sine transforms."""
    sx, lx, dx = _grid_axis(nx, peclet)
    sy, ly, dy = _grid_axis(ny, peclet)
    w = b.reshape(ny, nx) / (dy[:, None] * dx[None, :])
    w = (sy @ w @ sx) / (ly[:, None] + lx[None, :] - sigma)
    return ((sy @ w @ sx) * (dy[:, None] * dx[None, :])).reshape(-1)


def _normal(n, seed, k=None):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn((n,) if k is None else (k, n), generator=g, dtype=torch.float64, device=DEV)


def _torch_csr(csr):
    rowptr = torch.as_tensor(csr[0], device=DEV).long()
    rows = torch.repeat_interleave(torch.arange(len(csr[0]) - 1, device=DEV), rowptr[1:] - rowptr[:-1])
    return rows, torch.as_tensor(csr[1], device=DEV).long(), torch.as_tensor(csr[2], device=DEV).double()


def _mult(t, x, transpose=False):
    rows, cols, val = t
    if transpose:
        rows, cols = cols, rows
    return torch.zeros_like(x).index_add_(0, rows, val * x[cols])


def _arnoldi(t, v, steps, transpose=False, V=None, k=0):
    """Arnoldi with two full Gram-Schmidt passes, from v or from the rows 0..k of V: (V, H), a
    basis vector per row of V."""
    if V is None:
        V = torch.zeros((steps + 1, v.numel()), dtype=torch.float64, device=DEV)
        V[0] = v / v.norm()
    H = torch.zeros((k + steps + 1, k + steps), dtype=torch.float64, device=DEV)
    for j in range(k, k + steps):
        w = _mult(t, V[j], transpose)
        for _ in range(2):
            c = V[:j + 1] @ w
            w = w - c @ V[:j + 1]
            H[:j + 1, j] += c
        H[j + 1, j] = w.norm()
        V[j + 1] = w / H[j + 1, j]
    return V, H


class _Cuda:
    def __init__(self, ptr, shape, strides, typestr, owner):
        self.owner = owner      # the memory lives as long as a tensor over it
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": strides, "typestr": typestr,
                                         "version": 2}


def _view(owner, ptr, shape, strides, prec="f64"):
    """A tensor over the device memory of the library's object ``owner``."""
    size, typestr = (8, "<f8") if prec == "f64" else (4, "<f4")
    return torch.as_tensor(_Cuda(ptr, tuple(shape), tuple(s * size for s in strides), typestr, owner),
                           device=DEV)


def _vec_ptr(v):
    p = C.c_void_p()
    E._chk(E.lib().VecHIPGetArray(v, C.byref(p)), "VecHIPGetArray")
    return p.value


def _bv_columns(bv):
    """Device address of column 0 of a BV and its leading dimension (in bytes)."""
    at = []
    for j in (0, 1):
        v = C.c_void_p()
        E._chk(E.lib().BVGetColumn(bv.h, C.c_int(j), C.byref(v)), "BVGetColumn")
        at.append(_vec_ptr(v))
        E._chk(E.lib().BVRestoreColumn(bv.h, C.c_int(j), C.byref(v)), "BVRestoreColumn")
    return at[0], at[1] - at[0]


class _Default:
    """The default context of the framework as ks.Context names it, and torch on its stream."""

    def __init__(self):
        self.h = E.context_handle()
        self.stream = torch.cuda.ExternalStream(ks.lib().ks_ctx_stream(self.h))

    def sync(self):
        ks.check(ks.lib().ks_ctx_sync(self.h), "ks_ctx_sync")


_ctx = None


def _default():
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = _Default()
    return _ctx


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    ctx = _default()
    state = {"case": case, "ctx": ctx}
    globals()["_prepare_" + case["kind"]](state, case, int(seed))
    return state


def _prepare_solve(st, case, seed):
    csr = _matrix(case, seed)
    st["n"] = n = len(csr[0]) - 1
    st["A"] = E.Mat(csr)
    eps = st["eps"] = E.EPS()
    eps.setOperators(st["A"])
    eps.setProblemType(E.EPS.NHEP if case["matrix"] == "convdiff" else E.EPS.HEP)
    eps.setDimensions(case["nev"], case["ncv"])
    eps.setTolerances(1e-10)
    eps.setWhichEigenpairs(E.EPS.LARGEST_REAL if case["matrix"] == "convdiff" else E.EPS.LARGEST_MAGNITUDE)
    if case["twosided"]:
        eps.setTwoSided(True)
    if case["mixed"] > 0:
        eps.setMixedPrecision(case["mixed"])
    v0 = _normal(n, seed + 1).cpu().numpy()
    st["v0"] = E.Vec.from_array(v0)
    st["probe"] = torch.as_tensor(v0, device=DEV)
    # the vectors the eigenvectors go to, right ones first
    st["vecs"] = [E.Vec(n) for _ in range(case["nev"] * (2 if case["twosided"] else 1))]
    st["views"] = [_view(v, _vec_ptr(v.h), (n,), (1,)) for v in st["vecs"]]


def _requests(case, seed):
    reqs = M.serving_stream(case["requests"], 0.0, seed=seed, nmin=1000, nmax=case["nmax"])
    for i, r in enumerate(reqs):
        r["nev"] = 4 + (11 * i) % 29
        r["ncv"] = 2 * r["nev"] + 16
        r["csr"] = M.er_laplacian(r["n"], 8.0, seed=1000 * seed + i)
        r["v0"] = M.uniform_vector(seed + i, r["n"])
    return reqs


def _prepare_serve(st, case, seed):
    st["requests"] = _requests(case, seed)
    st["server"] = S.Server(4 << 30, 8)


def _krylov_basis(case, csr, seed):
    """k + 1 orthonormal rows of the Krylov basis, in the case's precision."""
    t = _torch_csr(csr)
    V, _ = _arnoldi(t, _normal(len(csr[0]) - 1, seed + 1), case["k"])
    return V.float() if case["prec"] == "f32" else V


def _prepare_expand(st, case, seed):
    csr = _matrix(case, seed)
    n, k, m = len(csr[0]) - 1, case["k"], case["k"] + case["steps"]
    size = 8 if case["prec"] == "f64" else 4
    st["A"] = E.Mat(csr)
    bv = st["bv"] = E.BV(n, m + 1, prec=E.F64 if case["prec"] == "f64" else E.F32)
    at, ld = _bv_columns(bv)
    V = _view(bv, at, (m + 1, n), (ld // size, 1), case["prec"])
    torch.cuda.synchronize()
    V[:k + 1] = _krylov_basis(case, csr, seed)
    torch.cuda.synchronize()
    st["H"], st["Hm"] = E.BV._dense(m + 1, m)
    st["new"] = V[k + 1:]
    st["args"] = (C.c_int(k), C.c_int(m), C.c_double(), C.c_int())


def _spmv_inputs(case, seed):
    csr = _matrix(case, seed)
    val = csr[2].astype(np.float32 if case["vprec"] == "f32" else np.float64)
    x = _normal(len(csr[0]) - 1, seed + 1)
    return (csr[0], csr[1], val), x if case["xprec"] == "f64" else x.float()


def _prepare_spmv(st, case, seed):
    csr, x = _spmv_inputs(case, seed)
    st["A"] = ks.CSR(st["ctx"], csr, prec=ks.F32 if case["vprec"] == "f32" else ks.F64)
    st["x"], st["y"] = x, torch.zeros_like(x)
    st["xprec"] = ks.F64 if case["xprec"] == "f64" else ks.F32


def _block_input(case, seed):
    """Columns that share a component, as the vectors of a subspace iteration do."""
    X = _normal(case["n"], seed, case["k"])
    X[1:] += 2.0 * X[0]
    return X


def _prepare_block(st, case, seed):
    bv = st["bv"] = E.BV(case["n"], case["k"])
    bv.set_block(BLOCKS[case["block"]])
    st["at"], ld = _bv_columns(bv)
    X = torch.zeros((case["k"], ld // 8), dtype=torch.float64, device=DEV)
    X[:, :case["n"]] = _block_input(case, seed)
    st["X"] = X
    st["Q"] = _view(bv, st["at"], (case["k"], case["n"]), (ld // 8, 1))


def _lu_shift(case, seed):
    """The middle of a wide gap near the middle of the grid operator's spectrum."""
    lx, ly = _grid_axis(case["nx"], 0.0)[1], _grid_axis(case["ny"], 0.0)[1]
    lam = torch.sort((ly[:, None] + lx[None, :]).reshape(-1))[0]
    mid = lam.numel() // 2 + seed % 7
    near = lam[max(0, mid - 30):mid + 30]
    gap = int(torch.argmax(near[1:] - near[:-1]))
    return float(0.5 * (near[gap] + near[gap + 1]))


def _prepare_lu(st, case, seed):
    n = case["nx"] * case["ny"]
    st["sigma"] = _lu_shift(case, seed)
    st["A"] = ks.CSR(st["ctx"], _grid(case["nx"], case["ny"], 0.0))
    st["b"] = _normal(n, seed, case["solves"])
    st["x"] = torch.zeros_like(st["b"])


def _p(t):
    return C.c_void_p(t.data_ptr())


def _prepare_inner(st, case, seed):
    n = case["nx"] * case["ny"]
    L, ctx = ks.lib(), st["ctx"]
    A = st["A"] = ks.CSR(ctx, _grid(case["nx"], case["ny"], case["peclet"]))
    st["b"] = _normal(n, seed)
    st["x"] = torch.zeros_like(st["b"])
    st["work"] = torch.zeros(6 * n + 64, dtype=torch.float64, device=DEV)
    torch.cuda.synchronize()
    if case["method"] == "bcgs-ilu":
        st["ilu"] = C.c_void_p()
        ks.check(L.ks_ilu0_create(ctx.h, A.h, C.c_double(0.0), C.byref(st["ilu"])), "ks_ilu0_create")
    else:
        st["dinv"] = torch.zeros_like(st["b"])
        torch.cuda.synchronize()
        ks.check(L.ks_pcg_jacobi(ctx.h, A.h, C.c_double(0.0), C.c_int(1), _p(st["dinv"])), "ks_pcg_jacobi")


# ------------------------------------------------------------------ run
def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _oriented(ctx, rows, probe):
    """Eigenvectors stacked, the sign of each fixed by the start vector."""
    with torch.cuda.stream(ctx.stream):
        X = torch.stack(rows)
        X *= torch.sign(X @ probe)[:, None]
    return X


def _run_solve(st):
    eps, nev = st["eps"], st["case"]["nev"]
    eps.setInitialSpace([st["v0"]])
    eps._keep.clear()
    eps.solve()
    if eps.getConverged() < nev:
        raise RuntimeError("the solve did not converge")
    lam = [eps.getEigenvalue(i) for i in range(nev)]
    L = E.lib()
    for i in range(nev):
        E._chk(L.EPSGetEigenvector(eps.h, C.c_int(i), st["vecs"][i].h, None), "EPSGetEigenvector")
    out = {"eigenvalues": np.array(lam), "X": _oriented(st["ctx"], st["views"][:nev], st["probe"])}
    if st["case"]["twosided"]:
        for i in range(nev):
            E._chk(L.EPSGetLeftEigenvector(eps.h, C.c_int(i), st["vecs"][nev + i].h, None), "EPSGetLeftEigenvector")
        out["Y"] = _oriented(st["ctx"], st["views"][nev:], st["probe"])
    return out


def _run_serve(st):
    srv = st["server"]
    ids = [srv.submit(r["csr"], r["nev"], r["ncv"], v0=r["v0"]) for r in st["requests"]]
    done = [None] * len(ids)
    while any(d is None for d in done):
        srv.progress()
        for i, rid in enumerate(ids):
            if done[i] is None:
                done[i] = srv.result(rid)
    return [d["eigr"] for d in done]


def _run_expand(st):
    k, m, beta, brk = st["args"]
    m = C.c_int(m.value)
    E._chk(E.lib().BVMatArnoldi(st["bv"].h, st["A"].h, st["Hm"], k, C.byref(m), C.byref(beta), C.byref(brk)),
           "BVMatArnoldi")
    return {"V": st["new"], "H": st["H"][:, k.value:m.value].copy(), "beta": beta.value}


def _run_spmv(st):
    ks.check(ks.lib().ks_spmv(st["ctx"].h, st["A"].h, _p(st["x"]), _p(st["y"]), st["xprec"], 0), "ks_spmv")
    return st["y"]


def _run_block(st):
    X, Q, ctx = st["X"], st["Q"], st["ctx"]
    ks.check(ks.lib().ks_memcpy_dtod(ctx.h, C.c_void_p(st["at"]), _p(X), X.numel() * 8), "ks_memcpy_dtod")
    R = st["bv"].orthogonalize()
    if st["case"]["block"].startswith("tsqr"):      # the QR with a positive diagonal, as Cholesky's
        s = np.where(np.diag(R) < 0, -1.0, 1.0)
        R *= s[:, None]
        with torch.cuda.stream(ctx.stream):
            Q *= torch.as_tensor(s, device=DEV)[:, None]
    return {"Q": Q, "R": R}


def _run_lu(st):
    L, ctx = ks.lib(), st["ctx"]
    F = ks.LU(ctx, st["A"], st["sigma"])
    for b, x in zip(st["b"], st["x"]):
        ks.check(L.ks_lu_solve(ctx.h, F.h, _p(b), _p(x)), "ks_lu_solve")
    F.check()
    F.close()
    return st["x"]


def _run_inner(st):
    L, ctx, method = ks.lib(), st["ctx"], st["case"]["method"]
    its, reason, rnorm = C.c_int(), C.c_int(), C.c_double()
    tail = (C.c_double(1e-11), C.c_double(0.0), C.c_int(20000), _p(st["work"]), C.byref(its), C.byref(rnorm),
            C.byref(reason))
    if method == "bcgs-ilu":
        e = L.ks_bcgs_solve_ilu(ctx.h, st["A"].h, C.c_double(0.0), st["ilu"], _p(st["b"]), _p(st["x"]), *tail)
    else:
        solve = L.ks_pcg_solve if method == "cg" else L.ks_bcgs_solve
        e = solve(ctx.h, st["A"].h, C.c_double(0.0), _p(st["dinv"]), _p(st["b"]), _p(st["x"]), *tail)
    ks.check(e, method)
    if reason.value <= 0:
        raise RuntimeError(f"{method} ended with reason {reason.value}")
    return st["x"]


# ------------------------------------------------------------------ work and tolerances
def _size(prec):
    return 8.0 if prec == "f64" else 4.0


def work(case):
    kind = case["kind"]
    if kind in ("solve", "serve"):
        if kind == "solve":
            jobs = [(_rows(case), _nnz(case), case["ncv"], 2 if case["twosided"] else 1)]
        else:   # the mean request of the stream: log-uniform sizes, nev 4 .. 32
            mean = (case["nmax"] - 1000) / math.log(case["nmax"] / 1000)
            jobs = [(mean, 9 * mean, 52, 1)] * case["requests"]
        b = f = 0.0
        for n, nnz, ncv, sides in jobs:
            steps = 3 * ncv     # a nominal four restarts of half the basis
            basis = 0.75 * ncv * n
            b += sides * steps * (12.0 * nnz + 20.0 * n + 2 * 8.0 * basis)
            f += sides * steps * (2.0 * nnz + 4.0 * basis)
        return {"bytes": b, "flops": f}
    if kind == "expand":
        n, s = _rows(case), _size(case["prec"])
        cols = sum(case["k"] + 1 + i for i in range(case["steps"]))
        return {"bytes": case["steps"] * (_nnz(case) * (s + 4.0) + n * (4.0 + 2 * s)) + 2.0 * cols * n * s,
                "flops": case["steps"] * 2.0 * _nnz(case) + 4.0 * cols * n}
    if kind == "spmv":
        return {"bytes": _nnz(case) * (_size(case["vprec"]) + 4.0) + _rows(case) * (4.0 + 2 * _size(case["xprec"])),
                "flops": 2.0 * _nnz(case)}
    if kind == "block":
        n, k = case["n"], case["k"]
        return {"bytes": 2 * 8.0 * n * k, "flops": 4.0 * n * k * k}
    n = case["nx"] * case["ny"]
    if kind == "lu":
        return {"bytes": 8.0 * n * n * (1 + case["solves"]), "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n * case["solves"]}
    its = 2.5 * case["nx"] if case["method"] == "cg" else (2.0 * case["nx"] if case["method"] == "bcgs" else 40.0)
    per = 5 * 12.0 + 8 * 11.0 if case["method"] == "cg" else 2 * 5 * 12.0 + 8 * 19.0
    return {"bytes": its * n * per, "flops": its * n * 40.0}


def tolerance(case):
    kind = case["kind"]
    if kind == "solve":     # pairs converged to 1e-10; a vector is as good as its gap lets it be
        return {"rel": 2e-6, "max": 5e-3}
    if kind == "serve":     # eigenvalues of symmetric pairs converged to 1e-10
        return {"rel": 1e-11, "max": 1e-10}
    if kind == "expand":    # a few steps of a recurrence that amplifies rounding
        return {"rel": 1e-12, "max": 1e-9} if case["prec"] == "f64" else {"rel": 2e-5, "max": 2e-3}
    if kind == "spmv":
        return {"rel": 4e-15, "max": 1e-12} if case["xprec"] == "f64" else {"rel": 2e-6, "max": 1e-4}
    if kind == "block":
        return {"rel": 1e-12, "max": 1e-10}
    if kind == "lu":
        return {"rel": 1e-10, "max": 1e-8}
    return {"rel": 2e-9, "max": 4e-8}     # an iteration stopped at 1e-11 of its first residual


# ------------------------------------------------------------------ exact
def exact(case, seed):
    seed = int(seed)
    kind = case["kind"]
    if kind == "solve":
        return _exact_solve(case, seed)
    if kind == "serve":
        return [_exact_pairs(_torch_csr(r["csr"]), torch.as_tensor(r["v0"], device=DEV), r["nev"], True)[0]
                for r in _requests(case, seed)]
    if kind == "expand":
        csr = _matrix(case, seed)
        k, m = case["k"], case["k"] + case["steps"]
        V = torch.zeros((m + 1, len(csr[0]) - 1), dtype=torch.float64, device=DEV)
        V[:k + 1] = _krylov_basis(case, csr, seed).double()
        V, H = _arnoldi(_torch_csr(csr), None, case["steps"], V=V, k=k)
        return {"V": V[k + 1:], "H": H[:, k:m].cpu().numpy(), "beta": float(H[m, m - 1])}
    if kind == "spmv":
        csr, x = _spmv_inputs(case, seed)
        return _mult(_torch_csr(csr), x.double())
    if kind == "block":
        Q, R = torch.linalg.qr(_block_input(case, seed).T.contiguous().cpu())
        s = torch.where(torch.diagonal(R) < 0, -1.0, 1.0).double()
        return {"Q": (Q * s).T.contiguous(), "R": (s[:, None] * R).numpy()}
    if kind == "lu":
        sigma = _lu_shift(case, seed)
        b = _normal(case["nx"] * case["ny"], seed, case["solves"])
        return torch.stack([_grid_solve(case["nx"], case["ny"], 0.0, sigma, v) for v in b])
    return _grid_solve(case["nx"], case["ny"], case["peclet"], 0.0, _normal(case["nx"] * case["ny"], seed))


def _exact_pairs(t, v0, nev, symmetric, transpose=False):
    """The nev rightmost (largest) eigenvalues and unit eigenvectors from one long Arnoldi run."""
    steps = min(v0.numel() - 1, 400)
    V, H = _arnoldi(t, v0, steps, transpose)
    H = H[:steps].cpu().numpy()
    if symmetric:
        lam, Z = np.linalg.eigh(0.5 * (H + H.T))
        order = np.argsort(-np.abs(lam))[:nev]
    else:
        lam, Z = np.linalg.eig(H)
        order = np.argsort(-lam.real)[:nev]
        lam, Z = lam.real, Z.real
    X = torch.as_tensor(np.ascontiguousarray(Z[:, order].T), device=DEV) @ V[:steps]
    return np.ascontiguousarray(lam[order]), X / X.norm(dim=1, keepdim=True)


def _exact_solve(case, seed):
    csr = _matrix(case, seed)
    t = _torch_csr(csr)
    v0 = _normal(len(csr[0]) - 1, seed + 1)
    lam, X = _exact_pairs(t, v0, case["nev"], case["matrix"] != "convdiff")
    out = {"eigenvalues": lam, "X": X * torch.sign(X @ v0)[:, None]}
    if case["twosided"]:
        Y = _exact_pairs(t, v0, case["nev"], False, True)[1]
        out["Y"] = Y * torch.sign(Y @ v0)[:, None]
    return out
