"""FP32 sweep with symmetric inverse blocks stored by their lower triangles: every packed block
size, cell counts around a workgroup's share, and a caller's matrix whose blocks are not
symmetric (which keeps the full blocks)."""
import numpy as np
import pytest

import bosss_amd as B
import oracle as O
from tests.helpers import log_uniform_nu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,k", [((3, 1), 3), ((13, 2), 3), ((8, 6), 3), ((5, 1), 4), ((9, 4), 4), ((3, 2, 1), 2),
                                     ((5, 5, 2), 2), ((1, 3, 1), 3), ((5, 3, 2), 3)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_sweep_blocks(ctx, shape, k, symmetric):
    print(f"case mg sym {shape} k={k} symmetric={symmetric}", flush=True)
    rng = np.random.default_rng(8)
    nodes = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.8, 1.2, n)) / n]) for n in shape]
    og = O.Grid(*nodes)
    nu = log_uniform_nu(og.J, 8)
    oo, go = O.Sip(og, k, nu), B.SipOperator(B.Grid(ctx, *nodes), k, nu)
    rp, col, val = oo.assemble()[0].export()
    val = val.copy()
    if not symmetric:   # a skew part of a tenth of the block's size
        for j in range(og.J):
            p = [q for q in range(rp[j], rp[j + 1]) if col[q] == j][0]
            s = rng.standard_normal(val[p].shape)
            val[p] += 0.1 * np.abs(val[p]).max() / oo.Np * (s - s.T)
    M = B.BlockMsrMatrix(ctx, nrows=og.J, bs=oo.Np, rowptr=rp, col=col, vals=val)
    b = rng.standard_normal(oo.N)
    out = []
    for prec in (B.BH_FP64, B.BH_FP32):
        mg = B.PMultigrid(go, M=M, degrees=[k, 1], min_coarse=1, omega=0.7, pre=1, post=1, kcycle_inner=0, prec=prec,
                          matrix_free=False)
        out.append(mg.Solve(np.zeros(oo.N), b))
    # matrix and inverse blocks are rounded to FP32: a sweep's error is a few unit roundoffs times
    # the blocks' condition (1e3 to 4e5 here; so with the full blocks)
    cond = max(np.linalg.cond(val[[q for q in range(rp[j], rp[j + 1]) if col[q] == j][0]]) for j in range(og.J))
    assert np.linalg.norm(out[1] - out[0]) <= 8 * 2.0 ** -24 * cond * np.linalg.norm(out[0])
