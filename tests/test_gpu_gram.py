"""The block dot Y^T X (ks_bv_gram): every count of 16-column tiles and its edges, more
than one 64 x 64 block, incomplete last rows, few rows, X and Y the same and not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("same", [True, False])
@pytest.mark.parametrize("n", [1, 15, 16, 63, 130, 1000, 70001])
def test_gram_tiles(prec, same, n):
    from slepc_amd import ks
    dt = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(n)
    ctx = ks.Context()
    ld = n + (n % 3)
    X = np.asfortranarray(rng.standard_normal((ld, 83)).astype(dt))
    Y = X if same else np.asfortranarray(rng.standard_normal((ld, 83)).astype(dt))
    dX = ks.DeviceArray.from_numpy(ctx, X)
    dY = dX if same else ks.DeviceArray.from_numpy(ctx, Y)
    x64, y64 = X[:n].astype(np.float64), Y[:n].astype(np.float64)
    ref = y64.T @ x64
    bound = 1.2e-16 * n * (np.abs(y64).T @ np.abs(x64)) + 1e-300   # any order of n products and sums
    sizes = [(p, p) for p in (1, 15, 16, 17, 33, 48, 49, 64, 65, 83)]
    if not same:
        sizes += [(1, 64), (64, 1), (17, 40), (40, 17), (80, 3), (33, 16), (50, 64)]
    for p, q in sizes:
        G = ks.DeviceArray.from_numpy(ctx, np.full((q + 2, p), 7.0, order="F"))
        ks.check(ks.lib().ks_bv_gram(ctx.h, prec, n, dX.ptr, ld, p, dY.ptr, ld, q, G.ptr, q + 2), "gram")
        g = G.numpy()
        assert (g[q:] == 7.0).all()
        assert (np.abs(g[:q] - ref[:q, :p]) <= bound[:q, :p]).all(), (p, q)
        if same:
            assert (g[:q] == g[:q].T).all()
    ctx.close()
