"""The inner CG and BiCGStab solves at the sizes where their launches change: one row
block, ragged blocks, the line between products that form their vector themselves
and those that read it, more row blocks than workgroups, and a row longer than a block."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _arrow(n):
    """Symmetric positive definite with a dense first row and column."""
    import scipy.sparse as sp
    A = sp.lil_matrix((n, n))
    A.setdiag(np.linspace(2.0, 3.0, n))
    A[0, 1:] = 0.01
    A[1:, 0] = 0.01
    A[0, 0] = 5.0
    A = A.tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data


def _cases():
    from slepc_amd import matgen as M
    yield M.laplacian_1d(1)
    yield M.laplacian_2d(17, 15)         # 255 rows: one ragged row block
    yield M.laplacian_2d(257, 1)
    yield M.laplacian_2d(301, 333)       # 99,965 rows, 498,557 entries: formed inside the product
    yield M.laplacian_2d(303, 333)       # 100,899 rows, 503,223 entries: formed before it
    yield M.laplacian_2d(901, 700)       # 630,700 rows: more row blocks than workgroups
    yield _arrow(3001)                   # a row longer than a block's entries


@pytest.mark.parametrize("method", ["pcg", "bcgs"])
@pytest.mark.parametrize("which", range(7))
def test_inner_solve(which, method):
    import scipy.sparse as sp
    from slepc_amd import ks
    csr = list(_cases())[which]
    n = len(csr[0]) - 1
    sigma = -0.05                        # condition number below 170 with the Laplacians' spectrum in (0, 8)
    ctx = ks.Context()
    L = ks.lib()
    A = ks.CSR(ctx, csr)
    b = np.random.default_rng(which).standard_normal(n)
    db, dx = ks.DeviceArray.from_numpy(ctx, b), ks.DeviceArray(ctx, n)
    work, dinv = ks.DeviceArray(ctx, 6 * n + 64), ks.DeviceArray(ctx, n)
    ks.check(L.ks_pcg_jacobi(ctx.h, A.h, C.c_double(sigma), C.c_int(1), dinv.ptr), "ks_pcg_jacobi")
    its, reason, rnorm = C.c_int(), C.c_int(), C.c_double()
    f = L.ks_pcg_solve if method == "pcg" else L.ks_bcgs_solve
    ks.check(f(ctx.h, A.h, C.c_double(sigma), dinv.ptr, db.ptr, dx.ptr, C.c_double(1e-11), C.c_double(0.0),
               C.c_int(2000), work.ptr, C.byref(its), C.byref(rnorm), C.byref(reason)), method)
    S = sp.csr_matrix((csr[2], csr[1], csr[0]), shape=(n, n)) - sigma * sp.identity(n)
    r = b - S @ dx.numpy()
    assert reason.value > 0
    # |B r| <= 1e-11 |B b|, B = diag^-1 within a factor 2.6 of a multiple of I; the recurrence's
    # residual drifts from the true one by a few eps times the iterations
    assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(b)
    A.free()
    ctx.close()
