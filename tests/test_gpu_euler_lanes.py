"""Euler right-hand side and time step at the edges of its lane and cell split: one to a few
cells per direction (every cell its own neighbour at one), cell counts below, at and above
what a wave and a workgroup take, every supported degree and quadrature, both precisions."""
import numpy as np
import pytest

import bosss_amd as B
import oracle as O
from test_gpu_euler import G, _say, _state

pytestmark = pytest.mark.gpu


def _grid(shape, seed):
    rng = np.random.default_rng(seed)
    return [np.concatenate([[0.0], np.cumsum(rng.uniform(0.8, 1.2, n)) / n]) for n in shape]


# cells per wave: 21 (3 lanes), 16 (4), 32 (2), 12 (5); four waves to a workgroup
CASES = [(D, k, q, s)
         for D, k, q, sizes in (
             (3, 1, 3, [(1, 1, 1), (3, 7, 4), (5, 17, 2)]),
             (3, 2, 4, [(1, 2, 3), (4, 4, 4), (13, 5, 1)]),
             (3, 1, 2, [(2, 1, 1), (3, 11, 4)]),
             (2, 2, 4, [(1, 1), (16, 4), (5, 13)]),
             (2, 3, 5, [(3, 1), (7, 7), (48, 1)]),
             (2, 1, 3, [(1, 5), (17, 5)]))
         for s in sizes]


@pytest.mark.parametrize("D,k,nq1,shape", CASES)
def test_rhs_and_stage_edges(ctx, D, k, nq1, shape):
    _say(f"case euler lanes D={D} k={k} nq1={nq1} {shape}")
    nodes = _grid(shape, 11)
    og = O.Grid(*nodes)
    oe = O.Euler(og, k=k, nq1=nq1, gamma=G)
    ge = B.EulerOperator(B.Grid(ctx, *nodes), k=k, nq1=nq1, gamma=G)
    U = _state(og, oe.Np, oe.nv, 12)
    ref = oe.rhs(U)
    # Scale of the terms that a coefficient adds up (they cancel where a cell is its own
    # neighbour): 2/h_d per direction, two faces, |p_j| <= sqrt(k + 1/2) at an end on the test
    # and on the trace side, (k + 1)^2 in all over the modes, and fluxes of the state's size.
    # The sums and a flux are some 60 operations deep, whose roundings add up as their root: 8
    # unit roundoffs of that scale
    terms = 2 * (k + 1) ** 2 * np.linalg.norm(U) * sum(2 / np.diff(x).min() for x in nodes)
    tol64, tol32 = 8 * 2.0 ** -53 * terms, 8 * 2.0 ** -24 * terms
    out = ge.rhs(U, np.zeros(ge.N))
    assert np.linalg.norm(out - ref) <= tol64
    # FP32, from arrays that are aligned to their elements only
    U32 = U.astype(np.float32)
    ref32 = oe.rhs(U32.astype(np.float64))
    dU = B.DeviceArray.from_host(ctx, np.concatenate([[0], U32]).astype(np.float32))
    dR = B.DeviceArray(ctx, ge.N + 1, np.float32)
    B._check(B.lib().bh_euler_rhs(ge.h, dU.ptr + 4, dR.ptr + 4, B.BH_FP32, B.BH_DEVICE_PTR))
    ctx.sync()
    out32 = dR.download()[1:].astype(np.float64)
    assert np.linalg.norm(out32 - ref32) <= tol32
    # two steps against the scheme in its textbook form
    h = 1e-3 / max(shape)
    refU = oe.tvd3(U, h, 2)
    outU = ge.tvd3(U.copy(), h, 2)
    assert np.linalg.norm(outU - refU) <= 16 * 2.0 ** -53 * np.linalg.norm(refU) + 2 * h * tol64


@pytest.mark.parametrize("D,k,nq1,shape", [(3, 2, 4, (4, 3, 5)), (2, 3, 5, (6, 7))])
@pytest.mark.parametrize("prec,root", [(B.BH_FP32, -75), (B.BH_FP32, 75), (B.BH_FP64, -600), (B.BH_FP64, 600)])
def test_size_of_the_cells(ctx, D, k, nq1, shape, prec, root):
    """The same flow on a grid 2^shift times the size: the coefficients scale with the root of
    the cells' volume, 2^root, the right-hand side by 2^-shift more, all by powers of two, so
    every bit but the exponents' is the same (the coefficients' squares leave the type's range)."""
    shift = 2 * root // D
    _say(f"case euler cell size D={D} prec={prec} shift={shift}")
    dt = np.float32 if prec == B.BH_FP32 else np.float64
    nodes = _grid(shape, 21)
    og = O.Grid(*nodes)
    U = None
    out = []
    for e in (0, shift):
        ge = B.EulerOperator(B.Grid(ctx, *[np.ldexp(a, e) for a in nodes]), k=k, nq1=nq1, gamma=G)
        if U is None:
            U = _state(og, ge.Np, D + 2, 22).astype(dt)
        dU = B.DeviceArray.from_host(ctx, np.ldexp(U, e * D // 2))
        dR = B.DeviceArray(ctx, ge.N, dt)
        ge.rhs(dU, dR, prec=prec)
        ctx.sync()
        dS = dU.download()
        ge.tvd3(dU, float(np.ldexp(1e-3, e)), 1, prec=prec)
        ctx.sync()
        out.append((np.ldexp(dR.download(), e - e * D // 2), np.ldexp(dU.download(), -e * D // 2)))
        assert np.array_equal(np.ldexp(dS, -e * D // 2), U)
    assert np.isfinite(out[0][0]).all()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("prec,rho,pressure", [(B.BH_FP32, 1e30, 1e-10), (B.BH_FP32, 1e38, 1.0), (B.BH_FP32, 5e-39, 1e-30),
                                               (B.BH_FP64, 1e305, 1e-5), (B.BH_FP64, 5.5e307, 1.0), (B.BH_FP64, 1e-308, 1e-200)])
@pytest.mark.parametrize("D,k,nq1,shape", [(3, 2, 4, (3, 4, 5)), (2, 3, 5, (6, 7))])
def test_ends_of_the_range(ctx, D, k, nq1, shape, prec, rho, pressure):
    """Gas at rest whose p / rho, density or inverse density is a denormal number (the
    hardware's approximate reciprocals and roots take it for zero)."""
    _say(f"case euler range D={D} prec={prec} rho={rho} p={pressure}")
    dt = np.float32 if prec == B.BH_FP32 else np.float64
    nodes = [2 * np.arange(n + 1.0) for n in shape]   # det J = 1
    og = O.Grid(*nodes)
    oe = O.Euler(og, k=k, nq1=nq1, gamma=G)
    ge = B.EulerOperator(B.Grid(ctx, *nodes), k=k, nq1=nq1, gamma=G)
    rng = np.random.default_rng(9)
    U = np.zeros((og.J, D + 2, ge.Np))
    U[:, 0, 0] = 2 ** (D / 2) * rho * rng.uniform(0.9, 1.0, og.J)
    U[:, D + 1, 0] = 2 ** (D / 2) * pressure / (G - 1) * rng.uniform(0.9, 1.0, og.J)
    U = U.astype(dt)
    ref = oe.rhs(U.astype(np.float64).ravel()).reshape(U.shape)
    assert np.isfinite(ref).all()
    dR = B.DeviceArray(ctx, ge.N, dt)
    ge.rhs(B.DeviceArray.from_host(ctx, U.ravel()), dR, prec=prec)
    ctx.sync()
    out = dR.download().reshape(U.shape).astype(np.float64)
    # a denormal number of 1e-40 (1e-310) has a unit of 1e-45 (5e-324): 1.4e-5 (5e-14) of it at
    # the input and in a quotient; a few of these per flux
    tol = 1e-4 if prec == B.BH_FP32 else 5e-13
    for v in range(D + 2):
        scale = np.abs(ref[:, v]).max()
        assert np.linalg.norm(out[:, v] / scale - ref[:, v] / scale) <= tol * np.linalg.norm(ref[:, v] / scale), v
