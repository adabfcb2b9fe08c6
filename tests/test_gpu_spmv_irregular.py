"""The product on matrices whose rows differ widely: rows longer than a row block (at its
multiples and remainders), long ones among short ones, empty rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = {"lengths": [2049, 2048, 2047, 0, 1, 4096, 4097, 6000, 16, 17, 33, 64, 65, 1000, 0],
        "short and long": ([3] * 200 + [40] + [900] + [2] * 50) * 3 + [5000],
        "one": [9000], "few": [700, 600, 500, 2100, 1], "none long": [2048, 5, 0, 2047, 1, 2048] + [3] * 300}


@pytest.mark.parametrize("vprec", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", list(ROWS))
def test_irregular_rows(kind, prec, vprec):
    from slepc_amd import ks
    lens = np.array(ROWS[kind])
    n, nc = len(lens), 9000
    rng = np.random.default_rng(n)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    colidx = np.concatenate([np.sort(rng.choice(nc, k, replace=False)) for k in lens]).astype(np.int32)
    val = rng.standard_normal(rowptr[-1]).astype(np.float64 if vprec == 0 else np.float32)
    dt = np.float64 if prec == 0 else np.float32
    x = rng.standard_normal(nc).astype(dt)
    ctx = ks.Context()
    A = ks.CSR(ctx, (rowptr, colidx, val), ncols=nc, prec=vprec)
    dx, dy = ks.DeviceArray.from_numpy(ctx, x), ks.DeviceArray.from_numpy(ctx, np.full(n, 7.0, dt))
    ks.spmv(ctx, A, dx, dy, prec)
    t = val.astype(np.float64) * x[colidx].astype(np.float64)
    ref = np.array([t[a:b].sum() for a, b in zip(rowptr[:-1], rowptr[1:])])
    mag = np.array([np.abs(t[a:b]).sum() for a, b in zip(rowptr[:-1], rowptr[1:])])
    eps = 2.3e-16 if prec == 0 else 1.2e-7   # each partial sum: at most a 256th of the row's entries and 14 more
    assert (np.abs(dy.numpy() - ref) <= eps * (lens / 64 + 40) * mag).all()
    A.free()
    ctx.close()
