"""Multigrid cycle with fused legs at its edges: block sizes 3 and 4, assembled and
matrix-free k = 1 levels, aggregates of one to eight cells (odd and one-cell directions), cell
counts around a wave's and a workgroup's share, one to three sweeps (the buffer that a leg
starts in alternates with their number), both precisions, with and without the K-cycle."""
import numpy as np
import pytest

import bosss_amd as B
import oracle as O
from tests.helpers import log_uniform_nu, nodes_3d

pytestmark = pytest.mark.gpu


def _nodes(shape, seed):
    if len(shape) == 3:
        return nodes_3d(*shape, jitter=0.3, seed=seed)
    rng = np.random.default_rng(seed)
    return [np.concatenate([[0.0], np.cumsum(rng.uniform(0.8, 1.2, n)) / n]) for n in shape]


@pytest.mark.parametrize("shape,k", [((9, 7, 5), 1), ((16, 8, 8), 1), ((1, 17, 3), 1), ((5, 4, 3), 2), ((33, 19), 1), ((16, 1), 1),
                                     ((9, 8), 2)])
@pytest.mark.parametrize("matrix_free", [False, True])
@pytest.mark.parametrize("pre,post", [(1, 1), (1, 2), (2, 2), (3, 1)])
def test_vcycle_edges(ctx, shape, k, matrix_free, pre, post):
    print(f"case mg legs {shape} k={k} mf={matrix_free} pre={pre} post={post}", flush=True)
    nodes = _nodes(shape, 3)
    og = O.Grid(*nodes)
    nu = log_uniform_nu(og.J, 3)
    oo = O.Sip(og, k, nu)
    go = B.SipOperator(B.Grid(ctx, *nodes), k, nu)
    Ao, _ = oo.assemble()
    b = np.random.default_rng(1).standard_normal(oo.N)
    degrees = [k, 1] if k > 1 else [1]
    ref, nl = Ao.pmg_vcycle(og, b, degrees, min_coarse=2, omega=0.7, pre=pre, post=post)
    assert nl >= 3
    # the smoother's and the coarsest level's inverses carry their blocks' condition: the bounds
    # of the same comparison at other sizes
    for prec, tol in ((B.BH_FP64, 1e-11), (B.BH_FP32, 1e-4)):
        mg = B.PMultigrid(go, degrees=degrees, min_coarse=2, omega=0.7, pre=pre, post=post, kcycle_inner=0, prec=prec,
                          matrix_free=matrix_free)
        for _ in range(3):   # eager, captured, replayed
            out = mg.Solve(np.zeros(oo.N), b)
            assert np.linalg.norm(out - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("n,matrix_free", [(128, False), (256, True)])
def test_block_array_on_a_page(ctx, n, matrix_free):
    """blocks of 3 in FP64 on a 128 x 128 level: 81,408 blocks of 72 bytes are 1,431 whole pages,
    so a column's load has nothing of its own behind the last block"""
    print(f"case mg legs page n={n} mf={matrix_free}", flush=True)
    nodes = _nodes((n, n), 4)
    og = O.Grid(*nodes)
    nu = log_uniform_nu(og.J, 4)
    oo = O.Sip(og, 1, nu)
    go = B.SipOperator(B.Grid(ctx, *nodes), 1, nu)
    b = np.random.default_rng(2).standard_normal(oo.N)
    ref, _ = oo.assemble()[0].pmg_vcycle(og, b, [1], min_coarse=64, omega=0.7, pre=1, post=1)
    mg = B.PMultigrid(go, degrees=[1], min_coarse=64, omega=0.7, pre=1, post=1, kcycle_inner=0, prec=B.BH_FP64,
                      matrix_free=matrix_free)
    out = mg.Solve(np.zeros(oo.N), b)
    assert np.linalg.norm(out - ref) <= 1e-11 * np.linalg.norm(ref)
