"""K-cycle's inner iteration at its edges: one to sixteen steps, vector lengths that are no
multiple of the 16-byte loads, lengths below and above a workgroup's share, a zero right-hand
side, both precisions."""
import numpy as np
import pytest

import bosss_amd as B
import oracle as O
from tests.helpers import log_uniform_nu
from tests.test_gpu_mg import _kcycle_numpy, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kin", [1, 2, 6, 16])
@pytest.mark.parametrize("shape", [(33, 19), (7, 5), (32, 24)])
def test_kcycle_steps(ctx, kin, shape):
    print(f"case kcycle kin={kin} {shape}", flush=True)
    kin = min(kin, 4) if shape == (7, 5) else kin   # a few steps solve the smallest system
    rng = np.random.default_rng(4)
    nodes = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.8, 1.2, n)) / n]) for n in shape]
    og = O.Grid(*nodes)
    nu = log_uniform_nu(og.J, 4)
    oo, go = O.Sip(og, 2, nu), B.SipOperator(B.Grid(ctx, *nodes), 2, nu)
    Ao, _ = oo.assemble()
    P = O.Pmg(Ao, og, [2, 1], min_coarse=8, omega=0.7, pre=1, post=1)
    b = rng.standard_normal(oo.N)
    # finest level: one sweep, truncation, K-cycle, one sweep
    rp, col, val = Ao.export()
    Np, J = oo.Np, og.J
    Dinv = np.array([np.linalg.inv(val[[p for p in range(rp[j], rp[j + 1]) if col[p] == j][0]]) for j in range(J)])
    A = lambda v: Ao.spmv(1.0, v, 0.0, np.zeros(oo.N))
    bj = lambda r: np.einsum("jab,jb->ja", Dinv, r.reshape(J, Np)).ravel()
    x = 0.7 * bj(b)
    xc = _kcycle_numpy(P, 1, (b - A(x)).reshape(J, Np)[:, :3].ravel(), kin)
    x = x.reshape(J, Np)
    x[:, :3] += xc.reshape(J, 3)
    x = x.ravel()
    x = x + 0.7 * bj(b - A(x))
    # the bounds of the same comparison at other sizes (FP64), and of an FP32 cycle
    for prec, tol in ((B.BH_FP64, 1e-9), (B.BH_FP32, 1e-3)):
        mg = B.PMultigrid(go, degrees=[2, 1], min_coarse=8, omega=0.7, pre=1, post=1, kcycle_inner=kin, prec=prec)
        for _ in range(3):   # eager, captured, replayed
            assert rel(mg.Solve(np.zeros(oo.N), b), x) < tol
        assert np.all(mg.Solve(np.zeros(oo.N), np.zeros(oo.N)) == 0.0)
