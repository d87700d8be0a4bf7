"""XDG evaluate against the assembled matrix on the device's own rules, where the split
into regular units and block rows can go wrong: grids of a few cells (no regular unit, one
partly filled wave), interfaces that reach the boundary, and level sets along grid planes
(cells without a cut whose neighbour lacks their species)."""
import numpy as np
import pytest

import bosss_amd as B

pytestmark = pytest.mark.gpu


def _problem(ctx, D, k, n, kind, graded=False):
    x = np.linspace(0, 1, n + 1)
    if graded:
        x = x ** 1.2
    g = B.Grid(ctx, *([x] * D))
    if kind == "sphere":
        return B.XdgPoisson(g, k, [0.5, 0.45, 0.52][:D], 0.3, 1.0, 1000.0)
    if kind == "boundary":
        return B.XdgPoisson(g, k, [0.1, 0.5, 0.5][:D], 0.33, 1.0, 1000.0)
    c = np.zeros((2,) * D)
    if kind == "plane":          # along the grid plane x = 1/2
        c[(0,) * D], c[(1,) + (0,) * (D - 1)] = -0.5, 1.0
    else:                        # tilted
        c[(0,) * D], c[(1,) + (0,) * (D - 1)], c[(0, 1) + (0,) * (D - 2)] = -0.62, 1.0, 0.31
    return B.XdgPoisson.poly(g, k, c, 1.0, 1000.0)


@pytest.mark.parametrize("D,k,n,kind,graded", [
    (2, 1, 3, "sphere", False), (2, 2, 4, "boundary", False), (2, 3, 5, "tilted", True), (2, 1, 8, "plane", False),
    (2, 2, 31, "sphere", True), (3, 1, 3, "sphere", False), (3, 2, 4, "boundary", True), (3, 1, 6, "plane", False),
    (3, 2, 7, "tilted", False), (3, 1, 17, "boundary", False), (3, 2, 13, "sphere", True)])
def test_evaluate_equals_assembled(ctx, D, k, n, kind, graded):
    print(f"case xdg evaluate vs assembled D={D} k={k} n={n} {kind} graded={graded}", flush=True)
    X = _problem(ctx, D, k, n, kind, graded)
    A = X.scipy_matrix(0)
    rng = np.random.default_rng(5)
    u, y0 = rng.standard_normal((2, X.N_full))
    ref = A @ u
    # both are sums of the same integrals: rounding of sums whose terms reach |A| |u|
    tol = 1e-13 * np.linalg.norm(abs(A) @ abs(u))
    out = X.Evaluate(1.0, 0.0, np.full(X.N_full, np.nan), u)
    assert np.linalg.norm(out - ref) <= tol
    out = X.Evaluate(-0.5, 2.0, y0.copy(), u)
    assert np.linalg.norm(out - (2.0 * y0 - 0.5 * ref)) <= tol
    d, r = B.DeviceArray.from_host(ctx, u), B.DeviceArray(ctx, X.N_full)
    X.Evaluate(1.0, 0.0, r, d)
    a = r.download()
    X.Evaluate(1.0, 0.0, r, d)
    assert np.array_equal(a, r.download())
