"""A whole expansion in one launch (ks_arnoldi_expand): one and several workgroups, both
ways of adding the dots and both register budgets at their lines, rows of many entries,
constraint columns, every refinement, FP64/FP32 data and values, breakdown, and the sizes it
leaves to the launches -- the relation A V = V H and the orthogonality in FP64 numpy."""
import ctypes as C

import numpy as np
import pytest

from slepc_amd import matgen as M

pytestmark = pytest.mark.gpu

EPS = {0: 2.3e-16, 1: 1.2e-7}


def _expand(csr, nc, k, m, prec=0, vprec=0, refine=0, seed=0, start=None, pad=0, launches=False):
    from slepc_amd import ks
    n = len(csr[0]) - 1
    dt = np.float64 if prec == 0 else np.float32
    ld = n + pad
    rng = np.random.default_rng(seed)
    Q = np.linalg.qr(rng.standard_normal((n, nc + 1)))[0]
    if start is not None:
        Q[:, nc] = start / np.linalg.norm(start)
    V = np.zeros((ld, nc + m + 1), dtype=dt, order="F")
    V[:n, :nc + 1] = Q
    ctx = ks.Context()
    A = ks.CSR(ctx, csr, prec=vprec)
    dV = ks.DeviceArray.from_numpy(ctx, V)
    ldb = nc + m + 2
    buf = ks.DeviceArray.from_numpy(ctx, np.zeros((ldb, m + 1), order="F"))
    taken = C.c_int(-1)
    out = []
    for a, b in ([(0, m)] if k == 0 else [(0, k), (k, m)]):
        ctx.status_reset()
        if launches:
            for j in range(a, b):
                ks.check(ks.lib().ks_spmv(ctx.h, A.h, dV.offset((nc + j) * ld), dV.offset((nc + j + 1) * ld), prec, 1),
                         "spmv")
                ks.check(ks.lib().ks_bv_orthonormalize_column(ctx.h, prec, n, dV.ptr, ld, nc + j + 1, buf.ptr, ldb, j + 1,
                                                              j + 1, refine, 0.7071, 1, 0), "column")
        else:
            ks.check(ks.lib().ks_arnoldi_expand(ctx.h, A.h, prec, n, dV.ptr, ld, nc, a, b, buf.ptr, ldb, refine, 0.7071,
                                                C.byref(taken)), "expand")
        out.append(ctx.status())
    r = dV.numpy(), buf.numpy(), out[-1], taken.value, A.info()["nblocks"]
    A.free()
    ctx.close()
    return r


def _dense_mul(csr, X, vprec):
    import scipy.sparse as sp
    v = np.asarray(csr[2], np.float64 if vprec == 0 else np.float32).astype(np.float64)
    return sp.csr_matrix((v, csr[1], csr[0]), shape=(len(csr[0]) - 1,) * 2) @ X


CASES = [  # matrix, its row blocks (workgroups), constraints, first, last column
    (lambda: M.convection_diffusion_2d(3), 1, 0, 0, 7),
    (lambda: M.convection_diffusion_2d(16), 1, 2, 0, 33),
    (lambda: M.convection_diffusion_2d(23), 3, 0, 5, 9),
    (lambda: M.er_laplacian(900, 40.0, 3), 19, 1, 0, 40),
    (lambda: M.convection_diffusion_2d(64), 16, 0, 16, 32),
    (lambda: M.convection_diffusion_2d(65), 17, 0, 16, 32),
    (lambda: M.convection_diffusion_2d(65), 17, 3, 0, 125),
    (lambda: M.convection_diffusion_2d(181), 128, 0, 0, 12),
    (lambda: M.convection_diffusion_2d(182), 130, 1, 4, 70),
    (lambda: M.convection_diffusion_2d(221), 191, 0, 0, 9),
]


@pytest.mark.parametrize("i", range(len(CASES)))
@pytest.mark.parametrize("prec,vprec,refine", [(0, 0, 0), (0, 1, 2), (1, 0, 0), (1, 1, 2), (0, 0, 1)])
def test_expansion_in_one_launch(i, prec, vprec, refine):
    make, blocks, nc, k, m = CASES[i]
    csr = make()
    n = len(csr[0]) - 1
    V, B, st, taken, nblocks = _expand(csr, nc, k, m, prec, vprec, refine, pad=i % 3)
    assert taken == 1 and nblocks == blocks and st.error == 0 and st.breakdown_col == -1
    assert (V[n:] == 0).all() and st.beta_last == B[nc + m, m]
    V = V[:n].astype(np.float64)
    H = B[:nc + m + 1, 1:m + 1]
    # A v_j = V h_j: rounding of the product (at most 60 entries a row) and of the nc + m term
    # updates, entrywise at most that many epsilons of norms up to |A|; FP32 data round w twice a pass
    anorm = np.abs(H).max() + 1e-300
    eps = EPS[max(prec, 0)] if vprec == 0 or prec == 1 else EPS[0]
    AV = _dense_mul(csr, V[:, nc:nc + m], vprec)
    assert np.abs(AV - V @ H).max() <= 8 * eps * np.sqrt(nc + m + 60) * anorm
    if refine != 1:   # two passes where needed: orthogonal to rounding, sums of n products
        G = V.T @ V - np.eye(nc + m + 1)
        assert np.abs(G).max() <= 8 * eps * np.sqrt(nc + m + 60)


@pytest.mark.parametrize("prec", [0, 1])
def test_same_coefficients_as_the_launches(prec):
    csr = M.er_laplacian(2000, 8.0, 1)
    a = _expand(csr, 1, 0, 12, prec)
    b = _expand(csr, 1, 0, 12, prec, launches=True)
    # twelve steps amplify a rounding of each sum by the ratios |A| / beta, under ten a step for this graph's
    # first ones together
    assert np.abs(a[1] - b[1]).max() <= 1e3 * EPS[prec] * np.abs(b[1]).max()
    for f in ("active", "breakdown_col", "col", "lindep", "error", "total_passes", "halt_col"):
        assert getattr(a[2], f) == getattr(b[2], f), f


@pytest.mark.parametrize("rows", [5, 40])
def test_breakdown_in_an_invariant_subspace(rows):
    n = 5000                                       # 20 workgroups; the start lives on the first rows only
    rng = np.random.default_rng(rows)
    S = rng.standard_normal((4, 4))
    r = np.concatenate([np.repeat(np.arange(4), 4), np.arange(4, n)])
    c = np.concatenate([np.tile(np.arange(4), 4), np.arange(4, n)])
    v = np.concatenate([S.ravel(), 1.0 + np.arange(4, n) / n])
    csr = (np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32), c.astype(np.int32), v)
    start = np.zeros(n)
    start[:4] = 1.0
    a = _expand(csr, 0, 0, rows, start=start)
    b = _expand(csr, 0, 0, rows, start=start, launches=True)
    assert a[3] == 1 and a[2].breakdown_col == b[2].breakdown_col == 4 and a[2].active == 0
    assert np.abs(a[1][:4, 1:4] - b[1][:4, 1:4]).max() <= 1e-12
    assert a[1][4, 4] == 0.0 == b[1][4, 4]


def test_left_to_the_launches():
    long = M.er_laplacian(3000, 8.0, 1)
    assert _expand(M.convection_diffusion_2d(222), 0, 0, 4)[3] == 0     # 193 row blocks
    assert _expand(long, 0, 0, 129)[3] == 0                             # more than 128 columns
    assert _expand(long, 2, 0, 127)[3] == 0
    assert _expand(M.laplacian_1d(12), 0, 0, 12)[3] == 0                # every column of the space
    n = 2200                                                            # a row longer than a row block
    rp = np.concatenate([[0, n], n + np.arange(1, n)]).astype(np.int32)
    ci = np.concatenate([np.arange(n), np.arange(1, n)]).astype(np.int32)
    assert _expand((rp, ci, np.ones(2 * n - 1)), 0, 0, 4)[3] == 0


@pytest.mark.parametrize("side,blocks,nc", [(23, 3, 1), (65, 17, 0), (182, 130, 2)])
def test_wait_that_runs_out(side, blocks, nc):
    """Waits that give up at their second poll: the status says so, every workgroup leaves, column
    k and those before it stay, and the context's next expansion is that of a new context."""
    from slepc_amd import ks
    csr = M.convection_diffusion_2d(side)
    n, k, m = side * side, 3, 24
    L, ldb = ks.lib(), nc + m + 2
    V0 = np.zeros((n, nc + m + 1), order="F")
    V0[:, :nc + 1] = np.linalg.qr(np.random.default_rng(side).standard_normal((n, nc + 1)))[0]
    taken, out = C.c_int(), []
    for disturb in (False, True):
        ctx = ks.Context()
        A = ks.CSR(ctx, csr)
        assert A.info()["nblocks"] == blocks
        dV, buf = ks.DeviceArray.from_numpy(ctx, V0), ks.DeviceArray.from_numpy(ctx, np.zeros((ldb, m + 1), order="F"))

        def expand(a, b):
            ctx.status_reset()
            ks.check(L.ks_arnoldi_expand(ctx.h, A.h, 0, n, dV.ptr, n, nc, a, b, buf.ptr, ldb, 0, 0.7071, C.byref(taken)),
                     "expand")
            assert taken.value == 1
            return ctx.status()
        assert expand(0, k).error == 0
        if disturb:
            V, B = dV.numpy(), buf.numpy()
            ks.check(L.ks_ctx_expand_polls(ctx.h, 1), "polls")
            st = expand(k, m)
            assert st.error == -8 and st.active == 0
            assert np.array_equal(dV.numpy()[:, :nc + k + 1], V[:, :nc + k + 1])
            assert np.array_equal(buf.numpy()[:, :k + 1], B[:, :k + 1])
            ks.check(L.ks_ctx_expand_polls(ctx.h, 0), "polls")
        st = expand(k, m)
        assert st.error == 0 and st.breakdown_col == -1
        out.append((dV.numpy(), buf.numpy(), st.total_passes))
        A.free()
        ctx.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]) and out[0][2] == out[1][2]


@pytest.mark.parametrize("side,nc", [(23, 2), (65, 0)])
def test_expansion_again_by_the_launches(side, nc):
    """BVMatArnoldi whose one launch gives up returns what the launches give, bit for bit, in that
    expansion and in the basis' next one."""
    from slepc_amd import eps as E
    from slepc_amd import ks
    n, k, m = side * side, 9, 20
    rng = np.random.default_rng(side)
    start, cons = rng.standard_normal(n), rng.standard_normal((n, max(nc, 1)))
    A = E.Mat(M.convection_diffusion_2d(side))
    out = {}
    for form in ("one launch", "launches", "again"):
        bv = E.BV(n, m + 1)
        if nc:
            assert bv.insert_constraints(cons) == nc      # makes the basis' storage again
        E._chk(E.lib().BVHIPKSSetOneLaunch(bv.h, C.c_int(form != "launches")), "BVHIPKSSetOneLaunch")
        bv.set_columns((start / np.linalg.norm(start))[:, None])
        E._chk(E.lib().BVOrthonormalizeColumn(bv.h, C.c_int(0), C.c_int(0), None, None), "BVOrthonormalizeColumn")
        got = []
        try:
            ks.check(ks.lib().ks_ctx_expand_polls(E.context_handle(), int(form == "again")), "polls")
            for a, b in ((0, k), (k, m)):
                H, h = E.BV._dense(m + 1, m)
                mm, beta, brk = C.c_int(b), C.c_double(), C.c_int()
                E._chk(E.lib().BVMatArnoldi(bv.h, A.h, h, C.c_int(a), C.byref(mm), C.byref(beta), C.byref(brk)),
                       "BVMatArnoldi")
                assert mm.value == b and not brk.value
                got += [H[:, a:b].copy(), beta.value]
                E.lib().MatDestroy(C.byref(h))
        finally:
            ks.check(ks.lib().ks_ctx_expand_polls(E.context_handle(), 0), "polls")
        out[form] = got + [bv.get_columns()]
        bv.destroy()
    A.destroy()
    assert not np.array_equal(out["one launch"][-1], out["launches"][-1])     # the sums of the two are ordered differently
    for a, b in zip(out["again"], out["launches"]):
        assert np.array_equal(a, b)


def test_context_rests_after_a_wait_that_ran_out():
    # 16 expansions by the launches, 32 after the next time-out
    from slepc_amd import ks
    csr, n = M.convection_diffusion_2d(65), 65 * 65
    ctx, L, taken = ks.Context(), ks.lib(), C.c_int()
    A = ks.CSR(ctx, csr)
    V = ks.DeviceArray.from_numpy(ctx, np.asfortranarray(np.random.default_rng(0).standard_normal((n, 31))))
    buf = ks.DeviceArray.from_numpy(ctx, np.zeros((32, 31), order="F"))

    def expand():
        ctx.status_reset()
        ks.check(L.ks_arnoldi_expand(ctx.h, A.h, 0, n, V.ptr, n, 0, 0, 30, buf.ptr, 32, 0, 0.7071, C.byref(taken)), "expand")
        return ctx.status().error if taken.value else None

    def polls(k):
        ks.check(L.ks_ctx_expand_polls(ctx.h, k), "polls")
    polls(1)
    assert [expand() for _ in range(18 + 33)] == [-8] + 16 * [None] + [-8] + 32 * [None] + [-8]
    polls(0)
    assert expand() == 0                                   # setting the polls forgets it
    polls(1)
    assert [expand() for _ in range(18)] == [-8] + 16 * [None] + [-8]
    A.free()
    ctx.close()
