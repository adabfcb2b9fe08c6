"""Gram-Schmidt against more than 128 columns (the sweep of eight wavefronts): every column
split and both sides of its lines, ragged rows, FP64 and FP32 with aligned and odd strides,
the full and the lean sequence, against two CGS passes in numpy."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KS = [128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 319]


@pytest.mark.parametrize("prec,pad", [(0, 0), (0, 3), (1, 0), (1, 1)])
@pytest.mark.parametrize("k", KS)
def test_wide_orthonormalization(k, prec, pad):
    from slepc_amd import ks
    n = 2 * k + 64 * (k % 5) + 7
    ld = (n + 1) // 2 * 2 + pad          # pad 1 with FP32: no row pairs
    dt = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(k)
    Q = np.linalg.qr(rng.standard_normal((n, k)))[0].astype(dt)
    w = (Q.astype(np.float64) @ rng.standard_normal(k) * 3.0 + 0.3 * rng.standard_normal(n) / np.sqrt(n)).astype(dt)
    V = np.zeros((ld, k + 1), dtype=dt, order="F")
    V[:n, :k], V[:n, k] = Q, w
    ctx = ks.Context()
    out = []
    for lean in (0, 1):
        dV = ks.DeviceArray.from_numpy(ctx, V)
        buf = ks.DeviceArray.from_numpy(ctx, np.zeros((k + 2, 3), order="F"))
        ctx.status_reset()
        f = ks.lib().ks_bv_orthonormalize_column_lean if lean else ks.lib().ks_bv_orthonormalize_column
        ks.check(f(ctx.h, prec, n, dV.ptr, ld, k, buf.ptr, k + 2, 2, 2, 0, 0.7071, 1, 0), "orthonormalize")
        st = ctx.status()
        if lean and st.halt_col >= 0:    # a third pass: completed as the expansions do
            ks.check(ks.lib().ks_bv_orthonormalize_resume(ctx.h, prec, n, dV.ptr, ld, k, buf.ptr, k + 2, 2, 2, 0,
                                                          0.7071), "resume")
            st = ctx.status()
        out.append((dV.numpy(), buf.numpy(), st.beta_last, st.lindep))
    (a, ha, na, la), (b, hb, nb, lb) = out
    assert la == 0 and lb == 0
    assert (a == b).all() and (ha[:, 2] == hb[:, 2]).all() and na == nb    # the same bits either way
    assert (a[:, :k] == V[:, :k]).all() and (a[n:] == 0).all()
    x, h = w.astype(np.float64), np.zeros(k)
    for _ in range(2):
        c = Q.astype(np.float64).T @ x
        x -= Q.astype(np.float64) @ c
        h += c
    # rounding of k-term sums in the data's precision; the vector is 1/30 of w, so its error is 30 times w's
    eps = (2.2e-16 if prec == 0 else 6e-8) * np.sqrt(n) * 40
    assert np.abs(ha[:k, 2] - h).max() <= eps * np.abs(h).max()
    assert abs(na - np.linalg.norm(x)) <= 30 * eps * np.linalg.norm(x)
    assert np.linalg.norm(a[:n, k] - x / np.linalg.norm(x)) <= 30 * eps
    ctx.close()
