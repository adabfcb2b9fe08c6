"""TSQR at the sizes where its tree changes: one wavefront to eight a node, leaves of 64 to
256 rows, ragged last leaves (shorter than a block of columns too), one to five levels, and
the widest panel a workgroup's LDS holds.  Against LAPACK's QR with R's diagonal positive."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (64, 1), (65, 3), (129, 8), (200, 9), (1000, 16), (4097, 17), (3001, 32), (2500, 33), (20011, 40),
          (777, 64), (513, 65), (1153, 96), (96, 96), (524288 + 5, 8), (300000, 12)]


@pytest.mark.parametrize("form_q", [1, 0])
@pytest.mark.parametrize("n,k", SHAPES)
def test_tsqr_shape(n, k, form_q):
    from slepc_amd import ks
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, k))
    X[:, 1:] += 2.0 * X[:, :1]
    ld = n + 3
    ctx = ks.Context()
    host = np.zeros((ld, k), order="F")
    host[:n] = X
    V = ks.DeviceArray.from_numpy(ctx, host)
    R = np.zeros((k + 1, k), order="F")
    ks.check(ks.lib().ks_bv_tsqr(ctx.h, C.c_int(n), V.ptr, C.c_int(ld), C.c_int(k), C.c_int(form_q),
                                 R.ctypes.data_as(C.c_void_p), C.c_int(k + 1)), "ks_bv_tsqr")
    Q = V.numpy()
    assert (Q[n:] == 0.0).all()                  # rows between n and ld are not touched
    R = R[:k]
    assert (np.tril(R, -1) == 0.0).all()
    Qe, Re = np.linalg.qr(X)
    s, se = np.where(np.diag(R) < 0, -1.0, 1.0), np.where(np.diag(Re) < 0, -1.0, 1.0)
    # backward stable factorizations of the same panel: R agrees to eps times its condition number
    # (below 1e3 here; square panels of normals reach about 10 k) times sqrt(n k) roundings
    eps = 2.2e-16 * np.sqrt(n * k) * max(np.linalg.cond(X), 10.0)
    assert np.linalg.norm(s[:, None] * R - se[:, None] * Re) <= eps * np.linalg.norm(Re)
    if form_q:
        assert np.linalg.norm(Q[:n].T @ Q[:n] - np.eye(k)) <= 4e-15 * k * np.log2(n + 2)
        assert np.linalg.norm(Q[:n] @ R - X) <= 1e-14 * k * np.linalg.norm(X)
    else:
        assert (Q[:n] == X).all()
    ctx.close()


def test_tsqr_refuses_wider_panels():
    from slepc_amd import ks
    ctx = ks.Context()
    V = ks.DeviceArray.from_numpy(ctx, np.zeros((400, 97), order="F"))
    R = np.zeros((97, 97), order="F")
    assert ks.lib().ks_bv_tsqr(ctx.h, C.c_int(400), V.ptr, C.c_int(400), C.c_int(97), C.c_int(1),
                               R.ctypes.data_as(C.c_void_p), C.c_int(97)) == -1   # KS_ERR_ARG
    ctx.close()
