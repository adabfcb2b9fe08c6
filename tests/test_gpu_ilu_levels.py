"""ILU(0) applied by levels in one workgroup (k_ilu0_levels) and by waiting rows
(k_ilu0_sf): one application of the factors against the oracle's in every form of the
layout (steps of 64 to 1024 rows, two or four entries a row, ring wrap-around) and where it
does not apply, the same bits from both forms, the room the layout takes, and the
solution of BiCGStab + ILU(0) against a dense solve."""
import ctypes as C

import numpy as np
import pytest

from test_ilu_layout import CASES, layered, layout

pytestmark = pytest.mark.gpu


def _solve(csr, b, rtol=1e-12, maxits=2000, room=None):
    """x, iterations, outcome and B b; room: bytes of device memory for the factors."""
    from slepc_amd import ks
    ctx = ks.Context()
    L = ks.lib()
    n = len(csr[0]) - 1
    A = ks.CSR(ctx, csr)
    db, dx = ks.DeviceArray.from_numpy(ctx, b), ks.DeviceArray(ctx, n)
    work = ks.DeviceArray(ctx, 6 * n + 64)
    M, pool = C.c_void_p(), C.c_void_p()
    if room:
        ks.check(L.ks_pool_create(C.byref(pool), C.c_size_t(room), C.c_size_t(0)), "ks_pool_create")
        L.ks_pool_use.restype = C.c_void_p
        L.ks_pool_use(pool)
    try:
        code = L.ks_ilu0_create(ctx.h, A.h, C.c_double(0.0), C.byref(M))
    finally:
        if room:
            L.ks_pool_use(C.c_void_p())
    ks.check(code, "ks_ilu0_create")
    its, reason, rnorm = C.c_int(), C.c_int(), C.c_double()
    ks.check(L.ks_bcgs_solve_ilu(ctx.h, A.h, C.c_double(0.0), M, db.ptr, dx.ptr, C.c_double(rtol), C.c_double(0.0),
                                 C.c_int(maxits), work.ptr, C.byref(its), C.byref(rnorm), C.byref(reason)),
             "ks_bcgs_solve_ilu")
    x, Bb = dx.numpy(), work.numpy()[n:2 * n]
    L.ks_ilu0_destroy(M)
    if room:
        ks.check(L.ks_pool_destroy(pool), "ks_pool_destroy")     # refused while anything is held
    A.free()
    ctx.close()
    return x, its.value, reason.value, Bb


def _cases():
    from slepc_amd import matgen as M
    yield "one row", M.laplacian_1d(1)
    yield "tridiagonal", M.laplacian_1d(700)            # 700 levels of one row: the ring never wraps
    yield "tridiagonal, ring wraps", M.laplacian_1d(3000)
    yield "5 x 4 grid", M.laplacian_2d(5, 4)
    yield "300 x 7 grid", M.laplacian_2d(300, 7)
    yield "257 x 255 grid", M.laplacian_2d(257, 255)    # widest level 255
    yield "258 x 257 grid", M.laplacian_2d(258, 257)    # widest level 257: steps of 512
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
    x, its, reason, _ = _solve(csr, b)
    assert reason > 0, (name, its, reason)
    # |B r| <= 1e-12 |B b|; the error is that times the preconditioned matrix' condition,
    # below 1e4 for these operators (the 257^2 Laplacian's own is 2.7e4, ILU(0) cuts it)
    xe = spl.spsolve(A.tocsc(), b) if n > 1 else b / A[0, 0]
    assert np.linalg.norm(x - xe) <= 1e-8 * np.linalg.norm(xe), name
    if name in ("one row", "tridiagonal", "tridiagonal, ring wraps", "wide levels", "wider levels"):
        assert its <= 3     # ILU(0) is the exact LU there


def _reference(csr, b):
    """(L U)^-1 b by substitution with the oracle's factors, and a bound of what another order or
    fused operations may differ by: with u the unit roundoff, (T + dT) x = b with |dT| <= m u |T|,
    and |T^-1| <= the inverse of T's comparison matrix.  m: the row's operations, 8 here, and as
    many again for the factors, which grow nothing in a diagonally dominant matrix."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl

    from oracle import oracle as O
    n = len(csr[0]) - 1
    F = sp.csr_matrix((O.ilu0(csr), csr[1], csr[0]), shape=(n, n))
    L, U = sp.tril(F, -1).tocsr() + sp.identity(n, format="csr"), sp.triu(F).tocsr()

    def solve(T, v, lower):
        return spl.spsolve_triangular(T.tocsr(), v, lower=lower)

    def compare(T):
        return (2 * sp.diags(np.abs(T.diagonal())) - abs(T)).tocsr()
    z = solve(L, b, True)
    y = solve(U, z, False)
    mu = 16 * 2.3e-16
    dz = solve(compare(L), mu * (abs(L) @ np.abs(z)), True)
    return y, solve(compare(U), mu * (abs(U) @ np.abs(y)) + dz, False)


@pytest.mark.parametrize("i", range(len(CASES)))
def test_one_application_of_the_factors(i):
    make, step, threads, entries = CASES[i]
    csr = make()
    n = len(csr[0]) - 1
    both = [layout(csr, lower) for lower in (1, 0)]
    assert all((L.step, L.threads, L.entries) == (step, threads, entries) for L in both)
    b = np.random.default_rng(i).standard_normal(n)
    Bb = _solve(csr, b, maxits=1)[3]
    y, bound = _reference(csr, b)
    assert (np.abs(Bb - y) <= bound).all()
    # without room for the layout the rows wait for each other: the same bits
    if step and n > 1000:
        factors = 4 * (n + len(csr[2]) + n) + 8 * len(csr[2]) + 16 * n + 2048       # ks_ilu0_create's other arrays
        less = factors + sum(L.bytes for L in both) // 2                            # its indices fit, not its values
        for room in (factors, less):
            assert np.array_equal(Bb, _solve(csr, b, maxits=1, room=room)[3])


def test_deep_levels_take_little_room():
    # a level a row: the factors and both layouts in under 1 KB a row
    from slepc_amd import matgen as M
    n = 20000
    csr = M.laplacian_1d(n)
    x, its, reason, _ = _solve(csr, np.ones(n), room=1000 * n)
    assert reason > 0 and its <= 3
    i = np.arange(1, n + 1)
    xe = 0.5 * i * (n + 1 - i)
    assert np.linalg.norm(x - xe) <= 1e-6 * np.linalg.norm(xe)    # condition 1.6e8
