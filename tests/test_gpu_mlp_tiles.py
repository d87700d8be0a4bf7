"""GPU parity of the network kernels at the edges of their cell tiles (inference: 16 cells,
four tiles per wave from 65,536 cells on; training: 32 cells, one workgroup per tile up to
256) and with arrays that are only float-aligned."""
import numpy as np
import pytest

import bosss_amd as B
from oracle import mlp as M

pytestmark = pytest.mark.gpu

WIDTHS = [(14, 6), (14, 20), (22, 10), (32, 20)]


def _net(ctx, n_in, n_out):
    """a network with non-zero biases (its own initialisation has none)"""
    net = B.CellMLP(ctx, n_in, n_out, seed=7)
    W1, b1, W2, b2, W3, b3 = M.unpack(net.get_params(), net.in_p, net.out_p)
    rng = np.random.default_rng(1)
    b3 = b3.copy()
    b3[:n_out] = 0.1 * rng.standard_normal(n_out)
    p = M.pack(W1, 0.1 * rng.standard_normal(128), W2, 0.1 * rng.standard_normal(128), W3, b3)
    net.set_params(p)
    return net, p


def _rows(n_in, n_in_p, rows, seed):
    X = np.zeros((rows, n_in_p), np.float32)
    X[:, :n_in] = np.random.default_rng(seed).standard_normal((rows, n_in))
    return X


def _off_kinks(p, X, in_p, out_p):
    """X with the rows that have a hidden unit within 1e-5 of its ReLU kink replaced: single
    precision (rounding about 1e-6 of a preactivation of order one) may put such a unit on
    the other side, and one unit moves a gradient of random signs by up to
    1 / sqrt(cells), not by rounding."""
    W1, b1, W2, b2, _, _ = [a.astype(np.float64) for a in M.unpack(p, in_p, out_p)]
    W1, W2 = M.bf16(W1).astype(np.float64), M.bf16(W2).astype(np.float64)
    a1 = X @ W1.T + b1
    a2 = np.maximum(a1, 0) @ W2.T + b2
    ok = np.minimum(np.abs(a1).min(1), np.abs(a2).min(1)) > 1e-5
    X = X.copy()
    X[~ok] = X[np.argmax(ok)]
    return X


def _at(ctx, a, offset):
    """device copy of a whose first element sits `offset` floats into an allocation"""
    d = B.DeviceArray(ctx, a.size + offset, np.float32)
    d.upload(np.concatenate([np.zeros(offset, np.float32), a.ravel()]))
    return d.view(offset, a.size), d


@pytest.mark.parametrize("n_in,n_out", WIDTHS)
@pytest.mark.parametrize("rows,offset", [(1, 0), (15, 0), (17, 1), (1000, 3), (65535, 0), (65536, 0), (65601, 1)])
def test_forward_tiles(ctx, n_in, n_out, rows, offset):
    print(f"case mlp forward tiles {n_in}->{n_out} rows {rows} offset {offset}", flush=True)
    net, p = _net(ctx, n_in, n_out)
    X = _rows(n_in, net.in_p, rows, 2)
    x, keep_x = _at(ctx, X, offset)
    y, keep_y = _at(ctx, np.full((rows, net.out_p), np.nan, np.float32), offset)
    net.forward(x, y)
    ctx.sync()
    Y = y.download().reshape(rows, net.out_p)
    assert np.all(Y[:, n_out:] == 0)
    # the oracle rounds the same values to BF16; a sum taken in another order may round a
    # hidden unit to the neighbouring BF16 value (2^-8 of it)
    ref = M.forward_infer(p, X, net.in_p, net.out_p)
    assert np.linalg.norm(Y - ref) <= 2e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("n_in,n_out", WIDTHS)
@pytest.mark.parametrize("rows,offset", [(1, 0), (31, 1), (33, 0), (8160, 0), (8161, 0), (8225, 1)])
def test_gradient_tiles(ctx, n_in, n_out, rows, offset):
    print(f"case mlp gradient tiles {n_in}->{n_out} rows {rows} offset {offset}", flush=True)
    net, p = _net(ctx, n_in, n_out)
    X = _off_kinks(p, _rows(n_in, net.in_p, rows, 3), net.in_p, net.out_p)
    T = _rows(n_out, net.out_p, rows, 4)
    x, keep_x = _at(ctx, X, offset)
    t, keep_t = _at(ctx, T, offset)
    loss, g = net.gradient(x, t)
    lref, gref = M.loss_grad(p, X, T, n_out, net.in_p, net.out_p, dtype=np.float64)
    # single precision sums: 32 terms of a tile, up to 2 tiles of a workgroup, 257 partials
    assert abs(loss - lref) <= 1e-6 * abs(lref)
    assert np.linalg.norm(g - gref) <= 1e-5 * np.linalg.norm(gref)
    # the targets as an upstream gradient, from the same device arrays
    gup = B.DeviceArray(ctx, net.n_params, np.float32)
    B._check(B.lib().bh_mlp_backward(net.h, rows, x.ptr, t.ptr, gup.ptr, B.BH_DEVICE_PTR))
    ctx.sync()
    uref = M.backward_upstream(p, X, T, n_out, net.in_p, net.out_p, dtype=np.float64)
    assert np.linalg.norm(gup.download() - uref) <= 1e-5 * np.linalg.norm(uref)
