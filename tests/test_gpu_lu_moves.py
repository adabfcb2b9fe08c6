"""The LU's row moves: pivots that lie anywhere below (a row-permuted diagonally dominant
matrix), in one panel, at its edge and over several with an incomplete last one."""
import numpy as np
import pytest

from slepc_amd import matgen as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [50, 128, 512, 513, 640, 1024, 1090, 1601])
@pytest.mark.parametrize("order", ["random", "reversed", "cyclic"])
def test_lu_of_permuted_rows(n, order):
    from slepc_amd import ks
    rng = np.random.default_rng(n)
    A = np.where(rng.random((n, n)) < 6.0 / n, rng.standard_normal((n, n)), 0.0) + 20.0 * np.eye(n)
    A = A[{"random": rng.permutation(n), "reversed": np.arange(n)[::-1], "cyclic": np.roll(np.arange(n), 77)}[order]]
    ctx = ks.Context()
    dA = ks.CSR(ctx, M.dense_to_csr(A))
    F = ks.LU(ctx, dA, 0.0)
    x = rng.standard_normal(n)
    db = ks.DeviceArray.from_numpy(ctx, A @ x)
    dx = ks.DeviceArray(ctx, (n,))
    F.solve(db, dx)
    F.check()
    # rows dominated by the pivot: no growth, a condition number of a few, sums of some ten terms
    assert np.abs(dx.numpy() - x).max() <= 100 * 2.3e-16 * 10 * np.abs(x).max()
    F.close()
    dA.free()
    ctx.close()
