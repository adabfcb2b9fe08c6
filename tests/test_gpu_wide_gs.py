"""Gram-Schmidt against more than 128 columns (the sweep of eight wavefronts): every column
split and both sides of its lines, ragged rows, FP64 and FP32 with aligned and odd strides,
the full and the lean sequence, against two CGS passes in numpy; and columns of 4 GiB and more,
whose rows need 64-bit offsets (k_gs_lds), against two passes in torch."""
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
    ld = (n + 1) // 2 * 2 + pad          # pad 1 with FP32: columns on 4-byte boundaries
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


@pytest.mark.parametrize("prec", [0, 1])
def test_columns_of_four_gib(prec):
    import torch

    from slepc_amd import ks
    n, k = (2 ** 29 if prec == 0 else 2 ** 30) + 77, 3
    ld = n + 1
    V = torch.zeros((k + 1, ld), dtype=torch.float64 if prec == 0 else torch.float32, device="cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    # orthonormal columns on every third row each, and a vector 0.05 away from their span
    for c in range(k):
        V[c, c:n:3] = torch.randn((n - c + 2) // 3, generator=g, dtype=V.dtype, device="cuda")
        V[c] /= torch.linalg.vector_norm(V[c], dtype=torch.float64).to(V.dtype)
    V[k, :n] = torch.randn(n, generator=g, dtype=V.dtype, device="cuda") * (0.05 / n ** 0.5)
    for c in range(k):
        V[k] += V[c] * (3.0, -2.0, 1.0)[c]
    x, h = V[k].to(torch.float64, copy=True), torch.zeros(k, dtype=torch.float64)
    for _ in range(2):
        q = [float((V[c].double() * x).sum()) for c in range(k)]
        onrm2 = float((x * x).sum())
        for c in range(k):
            x -= V[c].double() * q[c]
        x = x.to(V.dtype).double()
        h += torch.tensor(q, dtype=torch.float64)
    nrm = (onrm2 - sum(a * a for a in q)) ** 0.5
    torch.cuda.synchronize()
    ctx = ks.Context()
    buf = ks.DeviceArray.from_numpy(ctx, np.zeros((k + 2, 3), order="F"))
    ctx.status_reset()
    ks.check(ks.lib().ks_bv_orthonormalize_column_lean(ctx.h, prec, n, C.c_void_p(V.data_ptr()), ld, k, buf.ptr, k + 2, 2,
                                                       2, 0, 0.7071, 1, 0), "orthonormalize")
    st = ctx.status()
    assert st.halt_col < 0 and st.lindep == 0 and st.error == 0 and st.total_passes == 2
    hd = buf.numpy()[:, 2]
    # dots of FP64 products, summed 64 rows in turn in 2,049 sub-chunks at most, then 2,048 workgroups: under
    # 140,000 roundings in a row, 2e-11; the vector is 1/75 of w, its error as many times w's
    assert np.abs(hd[:k] - h.numpy()).max() <= 2e-11 * 3.8
    assert abs(hd[k] - nrm) <= 75 * 2e-11 * nrm and st.beta_last == hd[k]
    x /= nrm
    x -= V[k].double()
    err = float(torch.linalg.vector_norm(x))
    # FP32: the vector and the scaled vector are rounded once each
    assert err <= 75 * 2e-11 + (0 if prec == 0 else 1.2e-7)
    assert float(V[:, n].abs().max()) == 0
    ctx.close()
    del V, x
    torch.cuda.empty_cache()
