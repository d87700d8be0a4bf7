"""The calls a program makes of this library, as measurable cases.

Each case is one pass through the public Python mirror of the C ABI, with
device-resident vectors (``DeviceArray``), as a DG code that keeps its fields in
HBM calls it: operator evaluates, block-sparse products, multigrid cycles,
whole solves, the cut-cell operator, explicit Euler, and the learned
correction's network in both directions.

``path`` names the entry point, the other keys its sizes and options:

sip        ``SipOperator.Evaluate`` (form: apply, affine, residual)
spmv       ``BlockMsrMatrix.SpMV`` of the assembled operator
cycle      ``PMultigrid.Solve``: one preconditioner call
solve      ``FlexGMRES.Solve`` to 1e-8 with that preconditioner
xdg        ``XdgPoisson.Evaluate`` on cut cells
xdg_solve  ``XdgFlexGMRES.Solve`` to 1e-8 with its two-level preconditioner
euler      ``EulerOperator.rhs`` / one ``tvd3`` step
mlp        ``CellMLP.forward``
mlp_grad   ``CellMLP.gradient_noalloc`` (loss and parameter gradient)
"""
import math

import numpy as np
import torch

import bosss_amd as B

_CTX = None
_GAMMA = 1.4
_HID = 128


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = B.Context(0)
    return _CTX


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: the residual of a smooth source on 2D 64 x 64 quads, k = 2;
        # everything is in cache, so launches and latency are what it costs
        dict(name="sip2d_small", path="sip", D=2, nx=64, ny=64, nz=1, k=2, prec="f64", form="residual", grade=1.0, neumann=0),
        # the drop-in operator evaluate of a 3D Poisson problem, 5.2 M DOF
        dict(name="sip3d_f64", path="sip", D=3, nx=64, ny=64, nz=64, k=3, prec="f64", form="apply", grade=1.0, neumann=0),
        # a residual f - A u in single precision on a graded grid of odd sizes with mixed
        # boundary conditions: what a preconditioner's level computes
        dict(name="sip3d_f32_odd", path="sip", D=3, nx=51, ny=37, nz=45, k=2, prec="f32", form="residual", grade=1.01, neumann=5),
        # the assembled operator as BlockMsrMatrix (20 x 20 blocks): the drop-in's Krylov operator
        dict(name="spmv_f64", path="spmv", D=3, nx=64, ny=64, nz=64, k=3, prec="f64"),
        # one preconditioner call of the mixed-precision solver, log-uniform diffusion
        dict(name="cycle_f32", path="cycle", D=3, nx=64, ny=64, nz=64, k=3, prec="f32"),
        # a whole solve to 1e-8: log-normal diffusion, k = 2, single-precision multigrid
        dict(name="solve_f32", path="solve", D=3, nx=64, ny=64, nz=64, k=2, prec="f32"),
        # the cut-cell operator of the two-phase problem (sphere in 48^3, k = 2)
        dict(name="xdg_eval", path="xdg", D=3, n=48, k=2, cx=0.47, cy=0.53, cz=0.5, r=0.25),
        # a whole cut-cell solve to 1e-8, single-precision preconditioner
        dict(name="xdg_solve", path="xdg_solve", D=3, n=48, k=2, cx=0.47, cy=0.53, cz=0.5, r=0.25),
        # one time step of the explicit Euler solver, 44.2 M DOF: the largest state
        dict(name="euler_step_f64", path="euler", D=3, nx=96, ny=96, nz=96, k=2, prec="f64", form="step", grade=1.0),
        # a right-hand side in single precision on a graded grid of odd sizes
        dict(name="euler_rhs_f32_odd", path="euler", D=3, nx=47, ny=61, nz=35, k=2, prec="f32", form="rhs", grade=1.01),
        # the learned correction's inference over a whole grid (64^3 cells, k = 2 features)
        dict(name="mlp_forward", path="mlp", rows=262144, n_in=22, n_out=10),
        # its training pass on a slice of 32768 cells: loss and parameter gradient
        dict(name="mlp_grad", path="mlp_grad", rows=32768, n_in=22, n_out=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["sip", "sip", "sip", "spmv", "cycle", "solve", "xdg", "xdg", "xdg_solve", "euler", "euler", "mlp", "mlp_grad"])
    c = dict(path=path)
    if path == "sip":
        D = rng.choice([2, 3, 3])
        c.update(D=D, k=rng.randint(1, 4 if D == 2 else 3), prec=rng.choice(["f64", "f32"]))
        lo, hi = (16, 512) if D == 2 else (6, 72)
        c.update(nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi) if D == 3 else 1)
        # the affine part exists in double precision only
        c.update(form=rng.choice(["apply", "residual"] + (["affine"] if c["prec"] == "f64" else [])),
                 grade=rng.choice([1.0, 1.01]), neumann=rng.choice([0, 0, rng.randrange(1, 1 << (2 * D))]))
    elif path in ("spmv", "cycle", "solve"):
        k = rng.randint(1, 3) if path == "spmv" else rng.randint(2, 3)
        lo, hi = {"spmv": (6, 56), "cycle": (12, 56), "solve": (12, 48)}[path]
        c.update(D=3, k=k, prec=rng.choice(["f64", "f32"]))
        c.update(nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi))
    elif path in ("xdg", "xdg_solve"):
        D = rng.choice([2, 3, 3]) if path == "xdg" else 3
        c.update(D=D, n=_log_int(rng, 12, 48) if D == 3 else _log_int(rng, 20, 160), k=rng.randint(1, 3 if D == 2 else 2))
        c.update(cx=rng.uniform(0.4, 0.6), cy=rng.uniform(0.4, 0.6), cz=rng.uniform(0.4, 0.6), r=rng.uniform(0.2, 0.3))
    elif path == "euler":
        D = rng.choice([2, 3, 3])
        lo, hi = (16, 200) if D == 2 else (8, 80)
        c.update(D=D, k=rng.randint(1, 3 if D == 2 else 2), prec=rng.choice(["f64", "f32"]))
        c.update(nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi) if D == 3 else 1)
        c.update(form=rng.choice(["step", "rhs"]), grade=rng.choice([1.0, 1.01]))
    else:
        n_in, n_out = rng.choice([(14, 6), (22, 10), (32, 20), (16, 4)])
        c.update(rows=_log_int(rng, 500, 262144) if path == "mlp" else _log_int(rng, 200, 32768), n_in=n_in, n_out=n_out)
    return c


# ------------------------------------------------------------------ inputs
class _Mem:
    """A DeviceArray's memory for torch (no copy); keeps the array alive."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=(a.n,), typestr=a.dtype.str, data=(a.ptr, False), version=2)


def _t(a):
    return torch.as_tensor(_Mem(a), device="cuda")


def _array(t, dtype=np.float64):
    """A DeviceArray with the values of a torch tensor."""
    a = B.DeviceArray(_ctx(), t.numel(), dtype)
    _t(a).copy_(t.reshape(-1))
    return a


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(n, seed):
    return torch.randn(n, generator=_gen(seed), device="cuda", dtype=torch.float64)


def _np_dtype(case):
    return np.float32 if case["prec"] == "f32" else np.float64


def _prec(case):
    return B.BH_FP32 if case["prec"] == "f32" else B.BH_FP64


def _axis_nodes(n, grade):
    if grade == 1.0:
        return np.linspace(0.0, 1.0, n + 1)
    w = grade ** np.arange(n)
    return np.concatenate([[0.0], np.cumsum(w) / w.sum()])


def _nodes(c):
    return [_axis_nodes(c[a], c.get("grade", 1.0)) for a in ("nx", "ny", "nz")[:c["D"]]]


def _log_uniform_nu(J, seed):
    return 10.0 ** np.random.default_rng(seed).uniform(-2, 2, J)


def _log_normal_nu(c, seed, sigma=1.5, modes=16, ell=0.1):
    """exp(sigma g) at the cell centres, g a sum of random Fourier modes of correlation length ell."""
    rng = np.random.default_rng(seed)
    kv = torch.tensor(rng.normal(0.0, 1.0 / (2 * np.pi * ell), (modes, 3)), device="cuda")
    ph = torch.tensor(rng.uniform(0, 2 * np.pi, modes), device="cuda")
    g = 0
    xs = [torch.tensor(0.5 * (a[1:] + a[:-1]), device="cuda") for a in _nodes(c)]
    for m in range(modes):
        arg = (kv[m, 2] * xs[2])[:, None, None] + (kv[m, 1] * xs[1])[None, :, None] + (kv[m, 0] * xs[0])[None, None, :]
        g = g + torch.cos(2 * np.pi * arg + ph[m])
    return torch.exp(sigma * math.sqrt(2.0 / modes) * g).reshape(-1).cpu().numpy()


def _sine_coeffs(c, seed, modes=16, kmax=6):
    """DG coefficients of a sum of sine products with N(0,1) amplitudes (a smooth source)."""
    rng = np.random.default_rng(seed)
    D, k = c["D"], c["k"]
    ex = _exponents(D, k)
    xg, wg = np.polynomial.legendre.leggauss(8)
    L = _legendre(k, xg)[0] * wg[:, None]
    a = rng.standard_normal(modes)
    w = rng.integers(1, kmax + 1, (modes, D))
    out = 0
    for m in range(modes):
        S = []
        for d, x in enumerate(_nodes(c)):
            h = np.diff(x)
            X = x[:-1, None] + 0.5 * (xg + 1) * h[:, None]
            S.append(torch.tensor((np.sin(np.pi * w[m, d] * X) @ L * np.sqrt(h / 2)[:, None])[:, ex[:, d]], device="cuda"))
        if D == 3:
            out = out + a[m] * S[2][:, None, None] * S[1][None, :, None] * S[0][None, None]
        else:
            out = out + a[m] * S[0][:, None] * S[1][None]
    return out.reshape(-1)


def _euler_state(c, seed, modes=8, kmax=3, mach=0.2):
    """Conserved variables of a smooth periodic flow: density 1 + 0.1 Fourier modes, a
    divergence-free velocity at Mach 0.2, pressure 1/gamma, projected per cell."""
    D, k = c["D"], c["k"]
    rng = np.random.default_rng(seed)
    kv = rng.integers(-kmax, kmax + 1, (modes, D))
    kv[np.all(kv == 0, axis=1), 0] = 1
    A = rng.standard_normal(modes)
    A = 0.1 * A / np.abs(A).sum()
    ph, psi = rng.uniform(0, 2 * np.pi, (2, modes))
    if D == 3:
        dirs = np.cross(rng.standard_normal((modes, 3)), kv)
    else:
        dirs = np.stack([-kv[:, 1], kv[:, 0]], 1) * rng.standard_normal((modes, 1))
    dirs = mach * dirs / np.sqrt((dirs ** 2).sum(1)).sum()
    xg, wg = np.polynomial.legendre.leggauss(4)
    tab = _tables(D, k, xg, wg)
    xs = [torch.tensor(x[:-1, None] + 0.5 * (xg + 1) * np.diff(x)[:, None], device="cuda") for x in _nodes(c)]
    sc = _cell_volume(c, half=True).sqrt()
    PW = torch.tensor(tab["psi"] * tab["w"][:, None], device="cuda")
    lead = c["nz"] if D == 3 else c["nx"]
    step = max(1, 8 * 96 * 96 // max(1, (c["nx"] * c["ny"] if D == 3 else c["ny"])))
    out = []
    for s in range(0, lead, step):
        sl = slice(s, min(lead, s + step))
        if D == 3:
            X = [xs[0][None, None, :, :][..., tab["iq"][:, 0]], xs[1][None, :, None, :][..., tab["iq"][:, 1]],
                 xs[2][sl, None, None, :][..., tab["iq"][:, 2]]]
        else:
            X = [xs[0][sl, None, :][..., tab["iq"][:, 0]], xs[1][None, :, :][..., tab["iq"][:, 1]]]
        rho, u = 1.0, [0.0] * D
        for m in range(modes):
            arg = sum(2 * np.pi * float(kv[m, d]) * X[d] for d in range(D))
            rho = rho + A[m] * torch.sin(arg + ph[m])
            sn = torch.sin(arg + psi[m])
            u = [u[d] + dirs[m, d] * sn for d in range(D)]
        E = 1 / _GAMMA / (_GAMMA - 1) + 0.5 * rho * sum(v * v for v in u)
        F = torch.stack([rho] + [rho * v for v in u] + [E], -2)
        out.append((F @ PW) * sc[sl][..., None, None])
    return torch.cat(out).reshape(-1)


def _pad16(n):
    return (n + 15) // 16 * 16


def _mlp_params(c, seed):
    """W1, b1, W2, b2, W3, b3 (zero padding), He-uniform weights and small biases."""
    i, o = c["n_in"], c["n_out"]
    ip, op = _pad16(i), _pad16(o)
    rng = np.random.default_rng(seed)
    W1, W2, W3 = np.zeros((_HID, ip)), np.zeros((_HID, _HID)), np.zeros((op, _HID))
    W1[:, :i] = rng.uniform(-1, 1, (_HID, i)) * math.sqrt(6 / i)
    W2[:] = rng.uniform(-1, 1, (_HID, _HID)) * math.sqrt(6 / _HID)
    W3[:o] = rng.uniform(-1, 1, (o, _HID)) * math.sqrt(3 / _HID)
    b3 = np.zeros(op)
    b3[:o] = 0.1 * rng.standard_normal(o)
    p = [W1, 0.1 * rng.standard_normal(_HID), W2, 0.1 * rng.standard_normal(_HID), W3, b3]
    return [a.astype(np.float32) for a in p]


def _mlp_rows(c, seed):
    """Feature rows as the correction's feature map gives them: residual modes and
    neighbour residuals of unit norm, then logarithms of diffusion ratios."""
    r = torch.randn(c["rows"], c["n_in"], generator=_gen(seed + 1), device="cuda", dtype=torch.float32)
    own = c["n_in"] * 3 // 4
    X = torch.zeros(c["rows"], _pad16(c["n_in"]), device="cuda", dtype=torch.float32)
    X[:, :own] = r[:, :own] / r[:, :own].norm(dim=1, keepdim=True)
    X[:, own:c["n_in"]] = r[:, own:]
    return X


def _mlp_targets(c, seed):
    T = torch.zeros(c["rows"], _pad16(c["n_out"]), device="cuda", dtype=torch.float32)
    T[:, :c["n_out"]] = torch.randn(c["rows"], c["n_out"], generator=_gen(seed + 2), device="cuda", dtype=torch.float32)
    return T


# ------------------------------------------------------------------ prepare / run
class _State:
    pass


def _sip_op(c, nu):
    grid = B.Grid(_ctx(), *_nodes(c))
    bc = [(c.get("neumann", 0) >> f) & 1 for f in range(2 * c["D"])]
    return B.SipOperator(grid, c["k"], nu, bc=bc)


def _cells(c):
    return c["nx"] * c["ny"] * (c["nz"] if c["D"] == 3 else 1)


def _xdg(c):
    x = np.linspace(0.0, 1.0, c["n"] + 1)
    grid = B.Grid(_ctx(), *([x] * c["D"]))
    return B.XdgPoisson(grid, c["k"], [c["cx"], c["cy"], c["cz"]][:c["D"]], c["r"], 1.0, 1000.0, agg_threshold=0.1)


def _multigrid(c, op):
    return B.PMultigrid(op, degrees=[c["k"], 1], min_coarse=512, omega=0.8, pre=1, post=1, kcycle_inner=6, prec=_prec(c),
                        matrix_free=True)


def prepare(case, seed):
    c, s = case, _State()
    s.case = c
    ctx = _ctx()
    path = c["path"]
    if path == "sip":
        s.op = _sip_op(c, _log_uniform_nu(_cells(c), seed))
        dt = _np_dtype(c)
        if c["form"] == "affine":
            s.op.set_rhs(_array(_sine_coeffs(c, seed)))
        if c["form"] == "residual":
            s.f = _array(_sine_coeffs(c, seed), dt)
        s.u = _array(_randn(s.op.N, seed), dt)
        s.y = B.DeviceArray(ctx, s.op.N, dt)
        s.out = _t(s.y)
    elif path == "spmv":
        op = _sip_op(c, _log_uniform_nu(_cells(c), seed))
        s.M, _ = op.ComputeMatrix()
        dt = _np_dtype(c)
        s.u = _array(_randn(op.N, seed), dt)
        s.y = B.DeviceArray(ctx, op.N, dt)
        s.out = _t(s.y)
    elif path in ("cycle", "solve"):
        s.op = _sip_op(c, _log_uniform_nu(_cells(c), seed) if path == "cycle" else _log_normal_nu(c, seed))
        s.mg = _multigrid(c, s.op)
        if path == "solve":
            s.fg = B.FlexGMRES(op=s.op, Precond=s.mg, MaxKrylovDim=30, ConvergenceCriterion=1e-8, MaxSolverIterations=500)
        s.b = _array(_sine_coeffs(c, seed))
        s.zero = _array(torch.zeros(s.op.N, device="cuda", dtype=torch.float64))
        s.x = B.DeviceArray(ctx, s.op.N)
        s.out = _t(s.x)
    elif path == "xdg":
        s.X = _xdg(c)
        s.u = _array(_randn(s.X.N_full, seed))
        s.y = B.DeviceArray(ctx, s.X.N_full)
        s.out = _t(s.y)
    elif path == "xdg_solve":
        s.X = _xdg(c)
        rng = np.random.default_rng(seed)
        s.X.set_rhs(rng.uniform(0.5, 2.0, 2))
        s.P = B.XdgPrecond(s.X, prec=B.BH_FP32)
        B.xdg_precond_set_fp64_blocks(s.P, True)
        s.S = B.XdgFlexGMRES(s.X, s.P, MaxKrylovDim=30, ConvergenceCriterion=1e-8, MaxSolverIterations=1000)
        s.b = B.DeviceArray.from_host(ctx, s.X.rhs(1))
        s.zero = _array(torch.zeros(s.X.N, device="cuda", dtype=torch.float64))
        s.x = B.DeviceArray(ctx, s.X.N)
        s.out = _t(s.x)
    elif path == "euler":
        s.e = B.EulerOperator(B.Grid(ctx, *_nodes(c)), k=c["k"], nq1=_nq1(c), gamma=_GAMMA)
        s.dt = _euler_dt(c)
        s.U = _array(_euler_state(c, seed), _np_dtype(c))
        if c["form"] == "rhs":
            s.R = B.DeviceArray(ctx, s.e.N, _np_dtype(c))
        s.out = _t(s.U if c["form"] == "step" else s.R)
    else:
        s.net = B.CellMLP(ctx, c["n_in"], c["n_out"])
        s.net.set_params(np.concatenate([a.ravel() for a in _mlp_params(c, seed)]))
        s.x = _array(_mlp_rows(c, seed), np.float32)
        if path == "mlp":
            s.y = B.DeviceArray(ctx, c["rows"] * s.net.out_p, np.float32)
            s.out = _t(s.y)
        else:
            s.t = _array(_mlp_targets(c, seed), np.float32)
            s.grad = B.DeviceArray(ctx, s.net.n_params, np.float32)
            s.loss = B.DeviceArray(ctx, 1)
            s.out = (_t(s.grad), _t(s.loss))
    torch.cuda.synchronize()
    ctx.sync()
    return s


def run(state):
    s = state
    c = s.case
    path = c["path"]
    if path == "sip":
        if c["form"] == "residual":
            s.y.copy_from(s.f)
            s.op.Evaluate(-1.0, 1.0, s.y, s.u, affine=False, prec=_prec(c))
        else:
            s.op.Evaluate(1.0, 0.0, s.y, s.u, affine=c["form"] == "affine", prec=_prec(c))
    elif path == "spmv":
        s.M.SpMV(1.0, s.u, 0.0, s.y, prec=_prec(c))
    elif path == "cycle":
        s.x.copy_from(s.zero)
        s.mg.Solve(s.x, s.b)
    elif path == "solve":
        s.x.copy_from(s.zero)
        s.fg.Solve(s.x, s.b)
    elif path == "xdg":
        s.X.Evaluate(1.0, 0.0, s.y, s.u)
    elif path == "xdg_solve":
        s.x.copy_from(s.zero)
        s.S.Solve(s.x, s.b)
    elif path == "euler":
        if c["form"] == "step":
            s.e.tvd3(s.U, s.dt, 1, prec=_prec(c))
        else:
            s.e.rhs(s.U, s.R, prec=_prec(c))
    elif path == "mlp":
        s.net.forward(s.x, s.y)
    else:
        s.net.gradient_noalloc(s.x, s.t, s.grad, s.loss)
    return s.out


# ------------------------------------------------------------------ work and tolerance
def _modes(D, k):
    return math.comb(k + D, D)


def _sip_flops(c):
    D, k = c["D"], c["k"]
    Np, Nf = _modes(D, k), math.comb(k + D - 1, D - 1)
    nz = 0
    ex = _exponents(D, k)
    for d in range(D):
        o = [e for e in range(D) if e != d]
        same = (ex[:, None, o] == ex[None, :, o]).all(-1)
        nz += int((same & (ex[:, None, d] >= 1) & (ex[None, :, d] >= 1) & ((ex[:, None, d] + ex[None, :, d]) % 2 == 0)).sum())
    return _cells(c) * (2 * nz + D * (8 * (2 * Np - Nf) + 24 * Nf))


def work(case):
    c, path = case, case["path"]
    if path in ("sip", "spmv", "cycle", "solve"):
        Np, J = _modes(c["D"], c["k"]), _cells(c)
        N, e = J * Np, 4 if c["prec"] == "f32" else 8
        if path == "sip":
            return dict(bytes=N * e * (2 if c["form"] == "apply" else 3) + J * e, flops=_sip_flops(c))
        if path == "spmv":
            n = [c["nx"], c["ny"], c["nz"]]
            blocks = J + sum(2 * (J - J // n[d]) for d in range(3))
            return dict(bytes=blocks * (Np * Np * e + 4) + (J + 1) * 8 + 2 * N * e, flops=2 * blocks * Np * Np)
        # the vectors and the diffusion once; a cycle applies the finest operator 3 times and
        # the k = 1 operator 18 times (6 steps with 2 residuals and an apply each)
        coarse = dict(c, k=1)
        cyc = 3 * _sip_flops(c) + 18 * _sip_flops(coarse)
        its = 1 if path == "cycle" else 35
        return dict(bytes=2 * N * 8 + J * 8, flops=its * (cyc + (_sip_flops(c) if path == "solve" else 0)))
    if path in ("xdg", "xdg_solve"):
        D, k, n = c["D"], c["k"], c["n"]
        Np, J = _modes(D, k), n ** D
        area = 4 * math.pi * c["r"] ** 2 if D == 3 else 2 * math.pi * c["r"]
        cut = 1.5 * area * n ** (D - 1)
        N = (J + cut) * Np
        # the vectors, and per cut cell the element matrices of its volume, interface and face
        # items (about 22 blocks of Np x Np in 3D, 14 in 2D)
        em = cut * (22 if D == 3 else 14) * Np * Np
        if path == "xdg":
            return dict(bytes=2 * N * 8 + em * 8, flops=2 * em + _sip_flops(dict(D=D, k=k, nx=n, ny=n, nz=n)))
        return dict(bytes=2 * N * 8, flops=100 * 2 * N * 7 * Np)
    if path == "euler":
        D, k, q = c["D"], c["k"], _nq1(c)
        Np, NV, J = _modes(D, k), D + 2, _cells(c)
        N, e = J * NV * Np, 4 if c["prec"] == "f32" else 8
        # sum-factorised contractions: about q^D (k + 1) multiply-adds to the nodes and D times that
        # back per variable, a face mode expansion per face and side, the fluxes at the nodes
        vol = NV * 2 * q ** D * (k + 1) * (1 + D) + 30 * D * q ** D
        face = D * (NV * 4 * 2 * q ** (D - 1) * (k + 1) + 120 * q ** (D - 1))
        return dict(bytes=2 * N * e, flops=(3 if c["form"] == "step" else 1) * J * (vol + face))
    ip, op = _pad16(c["n_in"]), _pad16(c["n_out"])
    mac = ip * _HID + _HID * _HID + _HID * op
    n_params = mac + 2 * _HID + op
    if path == "mlp":
        return dict(bytes=c["rows"] * 4 * (ip + op) + n_params * 4, flops=2 * mac * c["rows"])
    return dict(bytes=c["rows"] * 4 * (ip + op) + n_params * 8, flops=6 * mac * c["rows"])


def tolerance(case):
    """About four times what the same path showed against 64 bits, or with another kernel
    form or precision of its parts, over the ranges of draw()."""
    c, path = case, case["path"]
    f32 = c.get("prec") == "f32"
    if path in ("sip", "spmv"):
        return {"rel": 5e-7, "max": 1.5e-5} if f32 else {"rel": 4e-15, "max": 1e-13}
    if path == "xdg":
        return {"rel": 1e-13, "max": 1e-11}
    if path == "cycle":
        return {"rel": 1.5e-5, "max": 3e-4} if f32 else {"rel": 1e-12, "max": 1e-10}
    if path in ("solve", "xdg_solve"):
        # the iterate at 1e-8 of the residual: one step more or fewer shows in the eighth digit
        return {"rel": 1e-8, "max": 1e-6}
    if path == "euler":
        if c["form"] == "step":
            return {"rel": 3e-7, "max": 2e-6} if f32 else {"rel": 1e-15, "max": 4e-15}
        # a right-hand side is the small difference of fluxes through opposite faces
        n = max(c["nx"], c["ny"], c["nz"])
        rel = min(0.03, 32 * (6e-8 if f32 else 1.1e-16) * n * n)
        return {"rel": rel, "max": min(0.9, 20 * rel)}
    if path == "mlp":
        return {"rel": 5e-3}   # activations in bfloat16
    return {"rel": 1e-6, "max": 1e-4}


# ------------------------------------------------------------------ 64-bit references
def _exponents(D, k):
    """Exponents per mode in the reference's mode order (degree, then x, then y exponent)."""
    ex = []
    for deg in range(k + 1):
        for a in range(deg + 1):
            ex += [(a, deg - a)] if D == 2 else [(a, b, deg - a - b) for b in range(deg - a + 1)]
    return np.array(ex)


def _legendre(k, x):
    """Orthonormal Legendre polynomials and derivatives on [-1, 1], each (len(x), k + 1)."""
    x = np.asarray(x, float)
    P, dP = np.zeros((len(x), k + 1)), np.zeros((len(x), k + 1))
    P[:, 0] = 1
    if k:
        P[:, 1], dP[:, 1] = x, 1
    for n in range(2, k + 1):
        P[:, n] = ((2 * n - 1) * x * P[:, n - 1] - (n - 1) * P[:, n - 2]) / n
        dP[:, n] = dP[:, n - 2] + (2 * n - 1) * P[:, n - 1]
    s = np.sqrt(np.arange(k + 1) + 0.5)
    return P * s, dP * s


def _tables(D, k, xg, wg):
    """Basis, gradients and weights at the tensor nodes; face traces per direction and side."""
    ex = _exponents(D, k)
    L, dL = _legendre(k, xg)
    E, _ = _legendre(k, [-1.0, 1.0])
    q = len(xg)
    iq = np.stack(np.meshgrid(*[np.arange(q)] * D, indexing="ij"), -1).reshape(-1, D)
    jq = np.stack(np.meshgrid(*[np.arange(q)] * (D - 1), indexing="ij"), -1).reshape(-1, D - 1)
    val = [L[iq[:, d]][:, ex[:, d]] for d in range(D)]
    grad = []
    for d in range(D):
        g = dL[iq[:, d]][:, ex[:, d]]
        for e in range(D):
            if e != d:
                g = g * val[e]
        grad.append(g)
    face = {}
    for d in range(D):
        other = [e for e in range(D) if e != d]
        for side in (0, 1):
            t = np.broadcast_to(E[side][ex[:, d]], (len(jq), len(ex)))
            for i, e in enumerate(other):
                t = t * L[jq[:, i]][:, ex[:, e]]
            face[d, side] = t
    return dict(iq=iq, w=np.prod(wg[iq], axis=1), psi=np.prod(val, axis=0), grad=grad, face=face, fw=np.prod(wg[jq], axis=1))


def _axis(D, d):
    """Tensor axis of direction d: cells are stored [z, y, x] in 3D and [x, y] in 2D."""
    return 2 - d if D == 3 else d


def _along(c, d, v):
    shape = [1] * c["D"]
    shape[_axis(c["D"], d)] = len(v)
    return torch.as_tensor(v, device="cuda", dtype=torch.float64).reshape(shape)


def _shape(c):
    return (c["nz"], c["ny"], c["nx"]) if c["D"] == 3 else (c["nx"], c["ny"])


def _cell_volume(c, half=False):
    v = 1
    for d, x in enumerate(_nodes(c)):
        v = v * _along(c, d, np.diff(x) * (0.5 if half else 1.0))
    return v.expand(_shape(c))


def _sip_exact(c, nu, u, penalty_base=1.3):
    """A u of the symmetric interior penalty operator, face by face."""
    D, k = c["D"], c["k"]
    ex = _exponents(D, k)
    Np = len(ex)
    nn = [c["nx"], c["ny"], c["nz"]][:D]
    h = [np.diff(x) for x in _nodes(c)]
    u = u.double().reshape(_shape(c) + (Np,))
    nu = torch.as_tensor(nu, device="cuda", dtype=torch.float64).reshape(_shape(c))
    pen = penalty_base * max((k + 1.0) * (k + D) / D, (k + 1.0) ** 2)
    cj = 0
    for d in range(D):
        nb = np.zeros(nn[d])
        nb[0] += 1
        nb[-1] += 1
        cj = cj + _along(c, d, (1 + 0.5 * nb) / h[d])
    cj = cj.expand(_shape(c))
    y = torch.zeros_like(u)
    xg, wg = np.polynomial.legendre.leggauss(k + 1)
    dL = _legendre(k, xg)[1]
    S = (dL * wg[:, None]).T @ dL
    E, dE = _legendre(k, [-1.0, 1.0])
    g = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    for d in range(D):
        o = [e for e in range(D) if e != d]
        same = (ex[:, None, o] == ex[None, :, o]).all(-1)
        Kd = g(np.where(same, S[ex[:, d]][:, ex[:, d]], 0.0))
        hd = _along(c, d, h[d]).expand(_shape(c))
        y -= (nu * 4 / hd ** 2)[..., None] * (u @ Kd.T)
        roots = np.where(ex[:, d] == 0)[0]
        F = same[:, roots]                       # mode -> face mode
        val = [g(F * E[s][ex[:, d]][:, None]) for s in (0, 1)]
        der = [g(F * dE[s][ex[:, d]][:, None]) for s in (0, 1)]
        ax = _axis(D, d)
        n = nn[d]
        P, Q = slice(0, n - 1), slice(1, n)
        at = lambda t, sl: t[tuple(sl if i == ax else slice(None) for i in range(D))]  # noqa: E731
        sc, gd = (2 / hd).sqrt(), 2 / hd
        if n > 1:
            nP, nQ, sP, sQ, gP, gQ = [at(t, w)[..., None] for t in (nu, sc, gd) for w in (P, Q)]
            uP, uQ = at(u, P), at(u, Q)
            AP, BP = uP @ val[1] * sP, uP @ der[1] * sP * gP
            AQ, BQ = uQ @ val[0] * sQ, uQ @ der[0] * sQ * gQ
            mu = pen * torch.maximum(at(cj, P), at(cj, Q))[..., None] * torch.maximum(nP, nQ)
            jump = AP - AQ
            flux = 0.5 * (nP * BP + nQ * BQ) - mu * jump
            at(y, P).add_((flux * sP) @ val[1].T + (0.5 * nP * jump * gP * sP) @ der[1].T)
            at(y, Q).add_((-flux * sQ) @ val[0].T + (0.5 * nQ * jump * gQ * sQ) @ der[0].T)
        for s in (0, 1):
            if (c.get("neumann", 0) >> (2 * d + s)) & 1:
                continue
            sl = slice(n - 1, n) if s else slice(0, 1)
            nP, sP, gP = [at(t, sl)[..., None] for t in (nu, sc, gd)]
            A, dn = at(u, sl) @ val[s] * sP, at(u, sl) @ der[s] * sP * gP * (1 if s else -1)
            mu = pen * at(cj, sl)[..., None]
            at(y, sl).add_(((nP * dn - 2 * mu * nP * A) * sP) @ val[s].T + (nP * A * gP * sP * (1 if s else -1)) @ der[s].T)
    return y.reshape(-1)


def _nq1(c):
    return {1: 3, 2: 4, 3: 5}[c["k"]]


def _euler_dt(c):
    return 0.3 * min(np.diff(x).min() for x in _nodes(c)) / ((2 * c["k"] + 1) * 1.2)


def _hllc(Ul, Ur, d, D):
    """HLLC flux in direction +d (pressure-based wave speeds) of conserved states [..., variable]."""
    g = _GAMMA

    def prim(U):
        rho, m, E = U[..., 0], U[..., 1:D + 1], U[..., D + 1]
        p = (g - 1) * (E - 0.5 * (m * m).sum(-1) / rho)
        return rho, m, E, m[..., d] / rho, p, torch.sqrt(g * p / rho)

    rl, ml, El, ul, pl, al = prim(Ul)
    rr, mr, Er, ur, pr, ar = prim(Ur)
    ps = (0.5 * (pl + pr) - 0.5 * (ur - ul) * 0.25 * (al + ar) * (rl + rr)).clamp(min=0)
    ql = torch.where(ps > pl, torch.sqrt(1 + (g + 1) / (2 * g) * (ps / pl - 1)), torch.ones_like(pl))
    qr = torch.where(ps > pr, torch.sqrt(1 + (g + 1) / (2 * g) * (ps / pr - 1)), torch.ones_like(pr))
    sl, sr = ul - al * ql, ur + ar * qr
    ss = (pr - pl + rl * ul * (sl - ul) - rr * ur * (sr - ur)) / (rl * (sl - ul) - rr * (sr - ur))
    left = ss > 0
    r, m, E = torch.where(left, rl, rr), torch.where(left[..., None], ml, mr), torch.where(left, El, Er)
    u, p, s = torch.where(left, ul, ur), torch.where(left, pl, pr), torch.where(left, sl, sr)
    F = torch.cat([(r * u)[..., None], m * u[..., None], (u * (E + p))[..., None]], -1)
    F[..., d + 1] += p
    star = torch.where(left, sl <= 0, sr >= 0)
    f = r * (s - u) / (s - ss)
    vel = m / r[..., None]
    vel[..., d] = ss
    Us = torch.cat([f[..., None], f[..., None] * vel, (f * (E / r + (ss - u) * (ss + p / (r * (s - u)))))[..., None]], -1)
    U = torch.cat([r[..., None], m, E[..., None]], -1)
    return torch.where(star[..., None], F + s[..., None] * (Us - U), F)


def _euler_rhs_exact(c, U, tab):
    D = c["D"]
    NV, Np = D + 2, _modes(D, c["k"])
    U = U.reshape(_shape(c) + (NV, Np))
    det = _cell_volume(c, half=True)
    sc = 1 / det.sqrt()
    h = [_along(c, d, np.diff(x)).expand(_shape(c)) for d, x in enumerate(_nodes(c))]
    g = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    R = torch.zeros_like(U)
    lead = U.shape[0]
    cells = det[0].numel()
    step = max(1, (1 << 17) // cells)
    psi, w = g(tab["psi"]), g(tab["w"])
    for s in range(0, lead, step):               # volume integrals, slab by slab
        sl = slice(s, s + step)
        Uq = (U[sl] @ psi.T) * sc[sl][..., None, None]
        rho, m, E = Uq[..., 0, :], Uq[..., 1:D + 1, :], Uq[..., D + 1, :]
        p = (_GAMMA - 1) * (E - 0.5 * (m * m).sum(-2) / rho)
        for d in range(D):
            v = m[..., d, :] / rho
            F = Uq * v[..., None, :]
            F[..., d + 1, :] += p
            F[..., D + 1, :] += p * v
            R[sl] += ((F * w) @ g(tab["grad"][d])) * (det[sl] * 2 / h[d][sl] * sc[sl])[..., None, None]
    for d in range(D):
        ax = _axis(D, d)
        fl, fr, fw = g(tab["face"][d, 1]), g(tab["face"][d, 0]), g(tab["fw"])
        Ul = ((U @ fl.T) * sc[..., None, None]).transpose(-1, -2)
        Ur = torch.roll(((U @ fr.T) * sc[..., None, None]).transpose(-1, -2), -1, ax)
        F = _hllc(Ul, Ur, d, D).transpose(-1, -2) * fw
        area = (det / (0.5 * h[d]))[..., None, None]
        R -= (F @ fl) * area * sc[..., None, None]
        R += (torch.roll(F * area, 1, ax) @ fr) * sc[..., None, None]
    return R.reshape(-1)


def exact(case, seed):
    c, path = case, case["path"]
    if path in ("sip", "spmv"):
        nu = _log_uniform_nu(_cells(c), seed)
        u = _randn(_cells(c) * _modes(c["D"], c["k"]), seed)
        if c["prec"] == "f32":
            # the operator as the single-precision path holds it: its inputs rounded once
            u = u.float()
        y = _sip_exact(c, nu, u)
        form = c.get("form", "apply")
        if form == "affine":
            y = y - _sine_coeffs(c, seed)
        if form == "residual":
            f = _sine_coeffs(c, seed)
            y = (f.float().double() if c["prec"] == "f32" else f) - y
        return y
    if path == "euler":
        U = _euler_state(c, seed)
        if c["prec"] == "f32":
            U = U.float().double()
        tab = _tables(c["D"], c["k"], *np.polynomial.legendre.leggauss(_nq1(c)))
        if c["form"] == "rhs":
            return _euler_rhs_exact(c, U, tab)
        dt = _euler_dt(c)
        k1 = _euler_rhs_exact(c, U, tab)
        k2 = _euler_rhs_exact(c, U + dt * k1, tab)
        k3 = _euler_rhs_exact(c, U + 0.25 * dt * (k1 + k2), tab)
        return U + dt / 6 * (k1 + k2 + 4 * k3)
    if path in ("mlp", "mlp_grad"):
        # the entry points round the weights to bfloat16 (the network as it is stored for inference)
        W1, b1, W2, b2, W3, b3 = [torch.tensor(a, device="cuda") for a in _mlp_params(c, seed)]
        W1, W2, W3 = [w.bfloat16().double() for w in (W1, W2, W3)]
        b1, b2, b3 = [b.double() for b in (b1, b2, b3)]
        X = _mlp_rows(c, seed).double()
        a1 = X @ W1.T + b1
        h1 = a1.clamp(min=0)
        a2 = h1 @ W2.T + b2
        h2 = a2.clamp(min=0)
        Y = h2 @ W3.T + b3
        if path == "mlp":
            return Y.reshape(-1)
        diff = Y - _mlp_targets(c, seed).double()
        diff[:, c["n_out"]:] = 0
        count = c["rows"] * c["n_out"]
        dY = 2 * diff / count
        d2 = (dY @ W3) * (a2 > 0)
        d1 = (d2 @ W2) * (a1 > 0)
        grad = torch.cat([t.reshape(-1) for t in (d1.T @ X, d1.sum(0), d2.T @ h1, d2.sum(0), dY.T @ h2, dY.sum(0))])
        return grad, (diff * diff).sum().reshape(1) / count
    return None   # solves, cycles and cut cells need the multigrid hierarchy or the cut-cell rules
