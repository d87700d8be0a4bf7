"""Block kernels at the edges of their load batches: block rows of none to twenty blocks (the
product of a row loads six columns per group at once), cell blocks of 3 to 40 rows (sixteen
lanes a block, ten columns at once), row counts around a workgroup's share."""
import numpy as np
import pytest
import scipy.linalg as sl

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


@pytest.mark.parametrize("Np", [3, 6, 10, 20])
@pytest.mark.parametrize("shape", [(3, 2), (7, 5)])
def test_cell_block_inverse(ctx, Np, shape):
    """Block-diagonal matrix of cells with one or two species: with omega = 1 and no sweep
    after it, the two-level preconditioner's first sweep is the solution and the coarse
    correction, of a residual of rounding size, is too."""
    print(f"case blocks inverse Np={Np} {shape}", flush=True)
    nodes = [np.linspace(0, 1, n + 1) for n in shape]
    g = B.Grid(ctx, *nodes)
    J = shape[0] * shape[1]
    rng = np.random.default_rng(Np)
    ln = Np * rng.integers(1, 3, J)
    i0 = np.concatenate([[0], np.cumsum(ln)[:-1]])
    blocks = []
    for n in ln:
        q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        blocks.append(q @ np.diag(rng.uniform(1.0, 4.0, n)) @ q.T)
    vals = np.concatenate([b.ravel() for b in blocks])
    M = B.BlockMsrMatrix.variable(ctx, np.arange(J + 1), np.arange(J), i0, ln, vals)
    b = rng.standard_normal(M.N)
    ref = sl.block_diag(*[np.linalg.inv(q) for q in blocks]) @ b
    # blocks of condition 4 and at most 40 rows: inverse, product, residual and correction
    for prec, eps, f64 in ((B.BH_FP64, 2.0 ** -53, 0), (B.BH_FP32, 2.0 ** -24, 0), (B.BH_FP32, 2.0 ** -24, 1)):
        P = B.XdgPrecondV(g, M, Np, coarse_degree=0, min_coarse=1, omega=1.0, pre=1, post=0, kcycle_inner=0, prec=prec)
        if f64:
            B.xdg_precond_set_fp64_blocks(P, True)
        out = P.Solve(np.zeros(M.N), b)
        assert np.linalg.norm(out - ref) <= 40 * 4 * 4 * eps * np.linalg.norm(b)
