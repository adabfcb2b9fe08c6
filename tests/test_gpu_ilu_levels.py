"""ILU(0) applied by levels in one workgroup (k_ilu0_levels) and by waiting rows
(k_ilu0_sf): the solution of BiCGStab + ILU(0) against a dense solve, at the sizes
where the level-ordered layout changes (steps of 256, 512 and 1024 rows, two or four
entries a row, ring wrap-around) and where it does not apply."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(csr, b, rtol=1e-12, maxits=2000):
    from slepc_amd import ks
    ctx = ks.Context()
    L = ks.lib()
    n = len(csr[0]) - 1
    A = ks.CSR(ctx, csr)
    db, dx = ks.DeviceArray.from_numpy(ctx, b), ks.DeviceArray(ctx, n)
    work = ks.DeviceArray(ctx, 6 * n + 64)
    M = C.c_void_p()
    ks.check(L.ks_ilu0_create(ctx.h, A.h, C.c_double(0.0), C.byref(M)), "ks_ilu0_create")
    its, reason, rnorm = C.c_int(), C.c_int(), C.c_double()
    ks.check(L.ks_bcgs_solve_ilu(ctx.h, A.h, C.c_double(0.0), M, db.ptr, dx.ptr, C.c_double(rtol), C.c_double(0.0),
                                 C.c_int(maxits), work.ptr, C.byref(its), C.byref(rnorm), C.byref(reason)),
             "ks_bcgs_solve_ilu")
    x = dx.numpy()
    L.ks_ilu0_destroy(M)
    A.free()
    ctx.close()
    return x, its.value, reason.value


def _cases():
    from slepc_amd import matgen as M
    yield "one row", M.laplacian_1d(1)
    yield "tridiagonal", M.laplacian_1d(700)            # 700 levels of one row: the ring never wraps
    yield "tridiagonal, ring wraps", M.laplacian_1d(3000)
    yield "5 x 4 grid", M.laplacian_2d(5, 4)
    yield "300 x 7 grid", M.laplacian_2d(300, 7)
    yield "257 x 255 grid", M.laplacian_2d(257, 255)    # widest level 255
    yield "258 x 257 grid", M.laplacian_2d(258, 257)    # widest level 257: steps of 1024
    yield "9^3 grid", M.varcoef_laplacian_3d(9)         # three entries a row
    yield "24^3 grid", M.varcoef_laplacian_3d(24)       # widest level beyond 256: steps of 512
    yield "graph", M.er_laplacian(1500, 8.0, seed=3)    # more entries than the layout takes
    yield "wide levels", _two_level(6000)               # three steps a level
    yield "wider levels", _two_level(9000)              # too wide for one workgroup


def _two_level(n):
    """Every second row depends on its neighbour: two levels thousands of rows wide."""
    i = np.arange(n)
    rowptr = np.zeros(n + 1, dtype=np.int32)
    rowptr[1:] = np.cumsum(np.where(i % 2 == 0, 1 + (i + 1 < n), 2))
    col, val = [], []
    for r in range(n):
        if r % 2 == 0:
            col += [r] + ([r + 1] if r + 1 < n else [])
            val += [4.0] + ([-1.0] if r + 1 < n else [])
        else:
            col += [r - 1, r]
            val += [-1.5, 5.0]
    return rowptr, np.array(col, dtype=np.int32), np.array(val)


@pytest.mark.parametrize("which", range(12))
def test_ilu_by_levels(which):
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl
    name, csr = list(_cases())[which]
    n = len(csr[0]) - 1
    A = sp.csr_matrix((csr[2], csr[1], csr[0]), shape=(n, n))
    if name == "graph":     # a graph Laplacian is singular: shift it
        A = (A + sp.identity(n)).tocsr()
        A.sort_indices()
        csr = (A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    b = np.random.default_rng(which).standard_normal(n)
    x, its, reason = _solve(csr, b)
    assert reason > 0, (name, its, reason)
    # |B r| <= 1e-12 |B b|; the error is that times the preconditioned matrix' condition,
    # below 1e4 for these operators (the 257^2 Laplacian's own is 2.7e4, ILU(0) cuts it)
    xe = spl.spsolve(A.tocsc(), b) if n > 1 else b / A[0, 0]
    assert np.linalg.norm(x - xe) <= 1e-8 * np.linalg.norm(xe), name
    if name in ("one row", "tridiagonal", "tridiagonal, ring wraps", "wide levels", "wider levels"):
        assert its <= 3     # ILU(0) is the exact LU there
