"""FP32 sweep with symmetric inverse blocks stored by their lower triangles: every packed block
size (10, 15 and 20 through the SIP hierarchy, 21, 28 and 35 through the coarse hierarchy of a
caller's variable-block matrix), cell counts around a workgroup's share, and a caller's matrix
whose blocks are not symmetric (which keeps the full blocks)."""
import math

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
        kept = "f64" if prec == B.BH_FP64 else "f32 triangles" if symmetric else "f32"
        assert B.pmg_level_blocks(mg) == kept
        out.append(mg.Solve(np.zeros(oo.N), b))
    # matrix and inverse blocks are rounded to FP32: a sweep's error is a few unit roundoffs times
    # the blocks' condition (1e3 to 4e5 here; so with the full blocks)
    cond = max(np.linalg.cond(val[[q for q in range(rp[j], rp[j + 1]) if col[q] == j][0]]) for j in range(og.J))
    assert np.linalg.norm(out[1] - out[0]) <= 8 * 2.0 ** -24 * cond * np.linalg.norm(out[0])


@pytest.mark.parametrize("shape,degree", [((5, 3), 5), ((4, 6), 5), ((3, 3), 6), ((8, 1), 6), ((3, 2, 1), 4), ((2, 2, 2), 4)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_sweep_blocks_of_a_callers_matrix(ctx, shape, degree, symmetric):
    D = len(shape)
    bs = math.comb(degree + D, D)
    print(f"case mg sym caller {shape} degree={degree} bs={bs} symmetric={symmetric}", flush=True)
    rng = np.random.default_rng(bs)
    g = B.Grid(ctx, *[np.linspace(0, 1, n + 1) for n in shape])
    J = int(np.prod(shape))
    # neighbours in the cells' numbering only: a chain, whatever the grid's faces are
    rp, col, blocks, cond = [0], [], [], 0
    off = [0.05 * rng.standard_normal((bs, bs)) / np.sqrt(bs) for _ in range(J - 1)]
    for r in range(J):
        for c in range(max(r - 1, 0), min(r + 2, J)):
            if c == r:
                q = np.linalg.qr(rng.standard_normal((bs, bs)))[0]
                d = q @ np.diag(rng.uniform(1.0, 4.0, bs)) @ q.T
                d = 0.5 * (d + d.T)
                if not symmetric:
                    s = rng.standard_normal((bs, bs))
                    d += 0.1 / bs * (s - s.T)
                cond = max(cond, np.linalg.cond(d))
                blocks.append(d)
            else:
                blocks.append(off[r] if c > r else off[c].T)
            col.append(c)
        rp.append(len(col))
    M = B.BlockMsrMatrix.variable(ctx, np.array(rp), np.array(col), bs * np.arange(J), np.full(J, bs),
                                  np.concatenate([a.ravel() for a in blocks]))
    b = rng.standard_normal(M.N)
    out = []
    for prec in (B.BH_FP64, B.BH_FP32):
        P = B.XdgPrecondV(g, M, bs, coarse_degree=degree, min_coarse=1, omega=0.7, pre=1, post=1, kcycle_inner=0, prec=prec)
        assert B.pmg_level_blocks(P) == ("f64" if prec == B.BH_FP64 else "f32 triangles" if symmetric else "f32")
        out.append(P.Solve(np.zeros(M.N), b))
    # as above, with blocks of condition 4: sweeps on both levels and the transfers between
    assert np.linalg.norm(out[1] - out[0]) <= 8 * 2.0 ** -24 * bs * cond * np.linalg.norm(out[0])
