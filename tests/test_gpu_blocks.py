"""Block kernels at the edges of their load batches: block rows of none to twenty blocks (the
product of a row loads six columns per group at once), row counts around a workgroup's share."""
import numpy as np
import pytest

import bosss_amd as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [8, 10, 15, 20, 21, 35])
@pytest.mark.parametrize("nrows", [1, 5, 22])
def test_spmv_row_lengths(ctx, bs, nrows):
    print(f"case blocks spmv bs={bs} nrows={nrows}", flush=True)
    rng = np.random.default_rng(bs * 100 + nrows)
    lens = [min(n, nrows) for n in (list(range(21)) + [7])[-nrows:]]
    rp = np.concatenate([[0], np.cumsum(lens)])
    col = np.concatenate([np.sort(rng.choice(nrows, n, replace=False)) for n in lens] + [np.zeros(0, int)]).astype(int)
    vals = rng.standard_normal((len(col), bs, bs))   # row-major blocks
    A = np.zeros((nrows * bs, nrows * bs))
    for r in range(nrows):
        for p in range(rp[r], rp[r + 1]):
            A[r * bs:(r + 1) * bs, col[p] * bs:(col[p] + 1) * bs] = vals[p]
    M = B.BlockMsrMatrix(ctx, nrows=nrows, bs=bs, rowptr=rp, col=col, vals=vals)
    x, y = rng.standard_normal(M.N), rng.standard_normal(M.N)
    # an entry adds at most 20 bs products
    scale = np.abs(A) @ np.abs(x) + np.abs(y)
    for beta in (0.0, -0.5):
        out = M.SpMV(2.0, x, beta, y.copy())
        assert np.all(np.abs(out - (2.0 * A @ x + beta * y)) <= 2 * 20 * bs * 2.0 ** -53 * scale + 1e-300)
        dx = B.DeviceArray.from_host(ctx, x.astype(np.float32))
        dy = B.DeviceArray.from_host(ctx, y.astype(np.float32))
        M.SpMV(2.0, dx, beta, dy, prec=B.BH_FP32)
        ctx.sync()
        assert np.all(np.abs(dy.download() - (2.0 * A @ x + beta * y)) <= 2 * (20 * bs + 3) * 2.0 ** -24 * scale + 1e-30)
