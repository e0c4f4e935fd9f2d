"""The work that users of this package have it do, as timed cases.

A case is one call of a solver's program into the package: an explicit run between two output times (the time
loop of an Euler or advection solver, restarted from a state kept on the device, then the field written back to
the host), one right-hand-side or limiter call through host memory (what a solver does that keeps its own time
loop), one implicit solve with its source and boundary data, and a batch of advection-diffusion cases.  The sizes
are those of the benchmark configurations and of the tests, with odd and ragged ones beside them.

Inputs come from the seed alone.  `exact` evaluates the same discretisations in plain 64-bit torch from their
definitions (nodes, operators, fluxes and time stepping written out below); of the package's files it reads only
the numbers of the triangle cubature rules, which are part of the scheme.
"""
import math
import os
import re

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GAMMA = 1.4
LSERK_A = (0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
           -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0)
LSERK_B = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0, 1720146321549.0 / 2090206949498.0,
           3134564353537.0 / 4481467310338.0, 2277821191437.0 / 14882151754819.0)
NQ = (0, 12, 19, 36, 54, 73, 93, 118, 145)   # cubature points of order N's rule


def listed():
    return [
        # the advection configuration: a Gaussian pulse, 2,048 elements; launches and latency count
        dict(name="advect_pulse_32x32_N4", kind="run", eq="advect", N=4, nx=32, ny=32, data="pulse", bc="periodic",
             flux="upwind", prec="fp64", scheme="lserk4", limiter="none", steps=20),
        # the isentropic-vortex tutorial: 1,024 elements, Roe flux, SSP-RK2, time-dependent inflow values
        dict(name="vortex_inflow_32x16_N4", kind="run", eq="euler", N=4, nx=32, ny=16, data="vortex", bc="inflow",
             flux="roe", prec="fp64", scheme="ssprk2", limiter="none", steps=20),
        # the headline benchmark: K = 131,072, order 6, FP64, the benchmark's 40 steps to the next output
        dict(name="vortex_256x256_N6", kind="run", eq="euler", N=6, nx=256, ny=256, data="vortex", bc="periodic",
             flux="lf", prec="fp64", scheme="lserk4", limiter="none", steps=40),
        # the same in its mixed-precision form with the learned troubled-cell indicator after every stage
        dict(name="vortex_256x256_N6_learned", kind="run", eq="euler", N=6, nx=256, ny=256, data="vortex",
             bc="periodic", flux="lf", prec="bf16x3", scheme="lserk4", limiter="mlp", steps=40),
        # an ordinary mid-size run in FP32; the element count is no multiple of 16
        dict(name="smooth_97x61_N6_fp32", kind="run", eq="euler", N=6, nx=97, ny=61, data="smooth", bc="periodic",
             flux="lf", prec="fp32", scheme="lserk4", limiter="none", steps=40),
        # a high-order run: order 8 on a small odd mesh
        dict(name="smooth_45x38_N8", kind="run", eq="euler", N=8, nx=45, ny=38, data="smooth", bc="periodic",
             flux="roe", prec="fp64", scheme="lserk4", limiter="none", steps=20),
        # the shock configuration with the reference driver's form: SSP-RK2, Roe, its Triangle limiter after each
        # stage (with the positivity scaling), open sides
        dict(name="shock_512x128_N3_triangle", kind="run", eq="euler", N=3, nx=512, ny=128, data="riemann", bc="open",
             flux="roe", prec="fp64", scheme="ssprk2", limiter="triangle", steps=20),
        # one right-hand side through host memory: a solver that keeps its own time loop hands the field over and
        # takes the derivative back
        dict(name="evaluate_63x50_N5", kind="evaluate", eq="euler", N=5, nx=63, ny=50, data="smooth", bc="periodic",
             flux="lf", prec="fp64"),
        # one limiter call through host memory, with the troubled-cell flags: such a solver's limiter hook
        dict(name="limit_131x77_N2", kind="limit", N=2, nx=131, ny=77, data="riemann", bc="open", limiter="tvb"),
        # the Poisson configuration: source and Dirichlet data from the host, FP64 block-Jacobi PCG, solution back
        dict(name="poisson_128x128_N5", kind="poisson", N=5, nx=128, ny=128, pc="block", mode="fp64", penalty="h",
             shift=0.0),
        # the viscous step of the projection solver on a small mesh: a Helmholtz solve of few iterations
        dict(name="helmholtz_40x33_N3", kind="poisson", N=3, nx=40, ny=33, pc="jacobi", mode="fp64",
             penalty="reference", shift=2000.0),
        # the ensemble configuration at 64 cases, orders 2..8, the whole step loop one captured graph
        dict(name="ensemble_64", kind="ensemble", cases=64, kmin=512, kmax=8192, nmin=2, nmax=8, draw=7, steps=20),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: meshes from a few elements to the largest listed ones, every order and
    option that the kinds above take."""
    kind = rng.choice(("run", "run", "run", "evaluate", "limit", "poisson", "poisson", "ensemble"))
    if kind == "ensemble":
        nmin = rng.randint(1, 6)
        return dict(kind=kind, cases=rng.randint(1, 64), kmin=64, kmax=_logint(rng, 256, 8192), nmin=nmin,
                    nmax=rng.randint(nmin, 8), draw=rng.randint(0, 10 ** 6), steps=rng.randint(3, 20))
    if kind == "poisson":
        N = rng.randint(1, 6)
        penalty = rng.choice(("h", "h", "reference"))   # the reference's is 20 times the other: more iterations
        n = (128 if N < 6 else 96) if penalty == "h" else 40
        nx, ny = _logint(rng, 3, n), _logint(rng, 3, n)
        shift = rng.choice((0.0, round(math.exp(rng.uniform(math.log(10.0), math.log(1e5))), 3)))
        return dict(kind=kind, N=N, nx=nx, ny=ny, pc=rng.choice(("jacobi", "block")),
                    mode=rng.choice(("fp64", "fp64", "mixed")), penalty=penalty, shift=shift)
    N = rng.randint(1, 8)
    n = 256 if N <= 6 else 160
    nx, ny = _logint(rng, 3, n), _logint(rng, 3, n)
    if kind == "limit":
        return dict(kind=kind, N=N, nx=nx, ny=ny, data="riemann", bc="open", limiter=rng.choice(("tvb", "triangle")))
    eq = rng.choice(("euler", "euler", "euler", "advect"))
    case = dict(kind=kind, eq=eq, N=N, nx=nx, ny=ny, data="pulse" if eq == "advect" else "smooth", bc="periodic",
                flux="upwind" if eq == "advect" else rng.choice(("lf", "roe")),
                prec=rng.choice(("fp64", "fp64", "fp32", "bf16x3")))
    if kind == "run":
        case.update(scheme=rng.choice(("lserk4", "ssprk2")), limiter="none", steps=rng.randint(2, 40))
        if eq == "euler" and rng.random() < 0.4:
            case.update(data="riemann", bc="open", flux="roe", prec="fp64", limiter=rng.choice(("tvb", "triangle")),
                        steps=rng.randint(2, 20))
    return case


# ---------------------------------------------------------------- the discretisation, written out
def _jacobi(x, a, b, n):
    """orthonormal Jacobi polynomial of degree n on [-1, 1] for the weight (1 - x)^a (1 + x)^b"""
    p0 = np.ones_like(x)
    p1 = 0.5 * ((a + b + 2) * x + (a - b))
    if n == 0:
        p = p0
    elif n == 1:
        p = p1
    else:
        for k in range(2, n + 1):   # the classical three-term recurrence
            c = 2 * k + a + b
            c1 = 2 * k * (k + a + b) * (c - 2)
            p0, p1 = p1, ((c - 1) * (c * (c - 2) * x + a * a - b * b) * p1
                          - 2 * (k + a - 1) * (k + b - 1) * c * p0) / c1
        p = p1
    norm = 2.0 ** (a + b + 1) / (2 * n + a + b + 1) * math.gamma(n + a + 1) * math.gamma(n + b + 1) / (
        math.factorial(n) * math.gamma(n + a + b + 1))
    return p / math.sqrt(norm)


def _djacobi(x, a, b, n):
    return np.zeros_like(x) if n == 0 else math.sqrt(n * (n + a + b + 1)) * _jacobi(x, a + 1, b + 1, n - 1)


def _basis(N, r, s):
    """orthonormal triangle basis and its r, s derivatives at (r, s): three arrays [points][Np]"""
    s1 = np.where(s < 1.0, 1.0 - s, 1.0)
    a = np.where(s < 1.0, 2.0 * (1.0 + r) / s1 - 1.0, -1.0)
    V, Vr, Vs = [], [], []
    h = 0.5 * (1.0 - s)
    for i in range(N + 1):
        for j in range(N - i + 1):
            f, g = _jacobi(a, 0, 0, i), _jacobi(s, 2 * i + 1, 0, j)
            df, dg = _djacobi(a, 0, 0, i), _djacobi(s, 2 * i + 1, 0, j)
            c = 2.0 ** (i + 0.5)
            hm = h ** (i - 1) if i > 0 else np.zeros_like(h)
            V.append(c * f * g * h ** i)
            vr = df * g * hm if i > 0 else np.zeros_like(h)
            Vr.append(c * vr)
            Vs.append(c * (0.5 * (1.0 + a) * vr + f * (dg * h ** i - 0.5 * i * g * hm)))
    return np.stack(V, 1), np.stack(Vr, 1), np.stack(Vs, 1)


def _lobatto(N):
    if N == 1:
        return np.array([-1.0, 1.0])
    c = np.zeros(N + 1)
    c[N] = 1.0
    inner = np.polynomial.legendre.legroots(np.polynomial.legendre.legder(c))
    x = np.concatenate([[-1.0], np.sort(inner.real), [1.0]])
    return 0.5 * (x - x[::-1])


def _nodes(N):
    """warp & blend nodes of the reference triangle (Warburton 2006)"""
    alpha = (0.0, 0.0, 1.4152, 0.1001, 0.2751, 0.98, 1.0999, 1.2832)[N - 1]
    L1 = np.array([(n - 1) / N for n in range(1, N + 2) for m in range(1, N + 3 - n)])
    L3 = np.array([(m - 1) / N for n in range(1, N + 2) for m in range(1, N + 3 - n)])
    L2 = 1.0 - L1 - L3
    eq = -1.0 + 2.0 * np.arange(N + 1) / N
    coef = np.linalg.solve(np.polynomial.legendre.legvander(eq, N), _lobatto(N) - eq)

    def warp(d):
        inside = np.abs(d) < 1.0 - 1e-10
        return np.where(inside, np.polynomial.legendre.legval(d, coef) / np.where(inside, 1.0 - d * d, 1.0), 0.0)

    w = [4 * L2 * L3 * warp(L3 - L2) * (1 + (alpha * L1) ** 2), 4 * L1 * L3 * warp(L1 - L3) * (1 + (alpha * L2) ** 2),
         4 * L1 * L2 * warp(L2 - L1) * (1 + (alpha * L3) ** 2)]
    x = L3 - L2 + w[0] + math.cos(2 * math.pi / 3) * w[1] + math.cos(4 * math.pi / 3) * w[2]
    y = (2 * L1 - L2 - L3) / math.sqrt(3.0) + math.sin(2 * math.pi / 3) * w[1] + math.sin(4 * math.pi / 3) * w[2]
    l1 = (math.sqrt(3.0) * y + 1.0) / 3.0
    l2 = (-3.0 * x - math.sqrt(3.0) * y + 2.0) / 6.0
    l3 = (3.0 * x - math.sqrt(3.0) * y + 2.0) / 6.0
    return l3 - l2 - l1, l1 - l2 - l3


def _fmask(N):
    """face nodes: face 0 along s = -1, face 1 the hypotenuse, face 2 along r = -1 back to the first vertex"""
    first = np.cumsum([0] + [N + 1 - i for i in range(N)])
    return np.stack([np.arange(N + 1), first + N - np.arange(N + 1), first[::-1]])


def _cubature(order):
    """the triangle rule of that order from the package's table of points and weights"""
    with open(os.path.join(ROOT, "hopefoam_amd", "csrc", "cubature_tri_table.inc")) as f:
        text = f.read()
    return [np.array([float(v) for v in re.search(r"dg_cub_%s%d\[\d+\] = \{([^}]*)\}" % (k, order), text).group(1)
                     .split(",")]) for k in "rsw"]


def _operators(N):
    r, s = _nodes(N)
    V, Vr, Vs = _basis(N, r, s)
    iV = np.linalg.inv(V)
    cr, cs, cw = _cubature(3 * (N + 1))
    Vc, Vcr, Vcs = _basis(N, cr, cs)
    Vq, Drq, Dsq = Vc @ iV, Vcr @ iV, Vcs @ iV
    M = Vq.T @ (cw[:, None] * Vq)
    iM = np.linalg.inv(M)
    gx, gw = np.polynomial.legendre.leggauss(N + 2)
    lg = _lobatto(N)
    Vf = np.linalg.solve(np.polynomial.legendre.legvander(lg, N).T, np.polynomial.legendre.legvander(gx, N).T).T
    fm = _fmask(N)
    E = np.zeros((len(r), 3, N + 2))
    En = np.zeros((len(r), 3, N + 1))
    for f in range(3):
        E[fm[f], f] += Vf.T * gw
        En[fm[f], f] += Vf.T @ (gw[:, None] * Vf)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    op = dict(r=r, s=s, Dr=Vr @ iV, Ds=Vs @ iV, Vq=Vq, Pr=iM @ (Drq.T * cw), Ps=iM @ (Dsq.T * cw), M=M, Vf=Vf, gw=gw,
              lift=iM @ E.reshape(len(r), -1), liftn=iM @ En.reshape(len(r), -1), Srr=Drq.T @ (cw[:, None] * Drq),
              Srs=Drq.T @ (cw[:, None] * Dsq), Sss=Dsq.T @ (cw[:, None] * Dsq))
    op = {k: torch.as_tensor(v, dtype=torch.float64, device=dev) for k, v in op.items()}
    op["fm"] = torch.as_tensor(fm, device=dev)
    return op


class _Mesh:
    """nx x ny split quads: quad (i, j) gives elements 2 (j nx + i) + {0, 1} with vertices (v00, v10, v11) and
    (v00, v11, v01); face k joins vertices k and k + 1; K x 3 neighbours (-1 at a boundary) and their faces"""

    def __init__(self, op, nx, ny, x0, x1, y0, y1, periodic):
        dev = op["r"].device
        K = 2 * nx * ny
        q = torch.arange(nx * ny, device=dev)
        i, j = q % nx, q // nx
        el = lambda ii, jj, t: 2 * ((jj % ny) * nx + ii % nx) + t  # noqa: E731
        nb = torch.stack([torch.stack([el(i, j - 1, 1), el(i + 1, j, 1), el(i, j, 1)], 1),
                          torch.stack([el(i, j, 0), el(i, j + 1, 0), el(i - 1, j, 0)], 1)], 1)
        nf = torch.tensor([[1, 2, 0], [2, 0, 1]], device=dev).expand(nx * ny, 2, 3)
        if not periodic:
            nb = nb.clone()
            nb[:, 0, 0][j == 0] = -1
            nb[:, 0, 1][i == nx - 1] = -1
            nb[:, 1, 1][j == ny - 1] = -1
            nb[:, 1, 2][i == 0] = -1
        self.K, self.nb, self.nf = K, nb.reshape(K, 3), nf.reshape(K, 3)
        hx, hy = (x1 - x0) / nx, (y1 - y0) / ny
        X, Y = x0 + i.double() * hx, y0 + j.double() * hy
        vx = torch.stack([torch.stack([X, X + hx, X + hx], 1), torch.stack([X, X + hx, X], 1)], 1).reshape(K, 3)
        vy = torch.stack([torch.stack([Y, Y, Y + hy], 1), torch.stack([Y, Y + hy, Y + hy], 1)], 1).reshape(K, 3)
        r, s = op["r"], op["s"]
        w = torch.stack([-0.5 * (r + s), 0.5 * (r + 1), 0.5 * (s + 1)])
        self.x, self.y = vx.double() @ w, vy.double() @ w
        t = torch.arange(K, device=dev) % 2   # the two shapes of the split quad
        xr, yr, xs, ys = torch.tensor([[hx, 0.0, hx, hy], [hx, hy, 0.0, hy]], dtype=torch.float64, device=dev)[t].T / 2
        self.J = xr * ys - xs * yr
        self.rx, self.ry, self.sx, self.sy = ys / self.J, -xs / self.J, -yr / self.J, xr / self.J
        nx_, ny_ = torch.stack([yr, ys - yr, -ys], 1), torch.stack([-xr, xr - xs, xs], 1)
        self.Js = torch.sqrt(nx_ * nx_ + ny_ * ny_)
        self.nx, self.ny = nx_ / self.Js, ny_ / self.Js
        self.fs = self.Js / self.J[:, None]
        inner = self.nb >= 0
        nbc = self.nb.clamp(min=0)
        self.fsmax = torch.where(inner, torch.maximum(self.fs, self.fs[nbc, self.nf]), self.fs)
        # nodes of the other side of each face, in the owner's order (boundary faces: the own nodes)
        fm = op["fm"]
        own = fm[None].expand(K, 3, -1) + (torch.arange(K, device=dev) * len(r))[:, None, None]
        other = fm[self.nf].flip(2) + (nbc * len(r))[:, :, None]
        self.own, self.inner = own, inner
        self.other = torch.where(inner[:, :, None], other, own)


def _vortex(x, y, p, t=0.0):
    """isentropic vortex of strength p[2] at (p[0] + t, p[1]) in the free stream (1, 0), r = squared distance"""
    dx, dy = x - p[0] - t, y - p[1]
    r = dx * dx + dy * dy
    rho = (1.0 - (GAMMA - 1.0) * p[2] ** 2 * torch.exp(2.0 * (1.0 - r)) / (16.0 * GAMMA * math.pi ** 2)) ** (
        1.0 / (GAMMA - 1.0))
    e = p[2] * torch.exp(1.0 - r) / (2.0 * math.pi)
    u, v = 1.0 - e * dy, e * dx
    return torch.stack([rho, rho * u, rho * v, rho ** GAMMA / (GAMMA - 1.0) + 0.5 * rho * (u * u + v * v)])


def _box(case):
    return {"pulse": (-1.0, 1.0, -1.0, 1.0), "riemann": (0.0, 2.0, 0.0, 0.5),
            "vortex": (0.0, 10.0, -5.0, 5.0), "smooth": (0.0, 10.0, 0.0, 10.0)}[case["data"]]


def _flow(case, seed):
    """operators, mesh and the initial state [vars][K][Np] of an explicit case, and the vortex's parameters"""
    rng = np.random.default_rng(seed)
    op = _operators(case["N"])
    mesh = _Mesh(op, case["nx"], case["ny"], *_box(case), periodic=case["bc"] == "periodic")
    x, y = mesh.x, mesh.y
    p = (5.0 + rng.uniform(-0.5, 0.5), rng.uniform(-0.5, 0.5), 5.0 * rng.uniform(0.9, 1.1))
    if case["data"] == "pulse":
        q = torch.exp(-40.0 * ((x - 0.3 * rng.uniform(-1, 1)) ** 2 + (y - 0.3 * rng.uniform(-1, 1)) ** 2))[None]
    elif case["data"] == "vortex":
        q = _vortex(x, y, p)
    elif case["data"] == "smooth":   # constant states with a few Fourier modes
        f = []
        for base, amp in ((1.0, 0.2), (0.3, 0.5), (-0.2, 0.5), (1.0, 0.2)):
            v = torch.full_like(x, base)
            for _ in range(3):
                kx, ky = (int(k) for k in rng.integers(1, 3, 2))
                v = v + amp / 3 * rng.uniform(-1, 1) * torch.sin(
                    2 * math.pi * (kx * x + ky * y) / 10.0 + rng.uniform(0, 2 * math.pi))
            f.append(v)
        q = torch.stack([f[0], f[0] * f[1], f[0] * f[2], f[3] / (GAMMA - 1) + 0.5 * f[0] * (f[1] ** 2 + f[2] ** 2)])
    else:                            # four-quadrant Riemann data
        xs, ys = rng.uniform(0.5, 1.5), rng.uniform(0.125, 0.375)
        st = np.stack([rng.uniform(0.2, 2.0, 4), rng.uniform(-1, 1, 4), rng.uniform(-1, 1, 4), rng.uniform(0.2, 2.0, 4)])
        quad = (x >= xs).long() + 2 * (y >= ys).long()
        rho, u, v, pr = (torch.as_tensor(st[k], device=x.device)[quad] for k in range(4))
        q = torch.stack([rho, rho * u, rho * v, pr / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)])
    return op, mesh, q, p


def _time_step(case, q):
    """CFL 0.4 (shocks 0.2) on the smallest node spacing and the inscribed circle"""
    x0, x1, y0, y1 = _box(case)
    hx, hy = (x1 - x0) / case["nx"], (y1 - y0) / case["ny"]
    if case["eq"] == "advect":
        speed = math.sqrt(2.0)
    else:
        u, v = q[1] / q[0], q[2] / q[0]
        pr = (GAMMA - 1) * (q[3] - 0.5 * q[0] * (u * u + v * v))
        speed = float((torch.sqrt(u * u + v * v) + torch.sqrt(GAMMA * pr / q[0])).max())
    spacing = float(np.diff(_lobatto(case["N"])).min())
    cfl = 0.2 if case["data"] == "riemann" else 0.4
    return cfl * 2.0 / 3.0 * spacing * hx * hy / (hx + hy + math.hypot(hx, hy)) / speed


# ---------------------------------------------------------------- the cases
def _case_nvar(case):
    return 1 if case.get("eq") == "advect" else 4


def _ensemble_cases(case):
    """like the ensemble configuration: K log-uniform, orders uniform, |a| in [0.5, 2], nu in [1e-3, 1e-2]"""
    rng = np.random.default_rng(case["draw"])
    out = []
    for _ in range(case["cases"]):
        n = max(3, int(round(math.sqrt(math.exp(rng.uniform(math.log(case["kmin"]), math.log(case["kmax"]))) / 2))))
        N = int(rng.integers(case["nmin"], case["nmax"] + 1))
        sp, th, nu, h = rng.uniform(0.5, 2.0), rng.uniform(0, 2 * math.pi), rng.uniform(1e-3, 1e-2), 1.0 / n
        dt = 0.5 * min(h / (sp * (N + 1) ** 2), h * h / (nu * (N + 1) ** 4))
        out.append(dict(N=N, nx=n, ny=n, x0=0.0, y0=0.0, Lx=1.0, Ly=1.0, ax=sp * math.cos(th), ay=sp * math.sin(th),
                        nu=nu, dt=dt))
    return out


def _ensemble_states(case, seed):
    """(case, operators, mesh, initial state [K][Np]) of every ensemble member"""
    rng = np.random.default_rng(seed)
    ops = {}
    for c in _ensemble_cases(case):
        op = ops.setdefault(c["N"], _operators(c["N"]))
        m = _Mesh(op, c["nx"], c["ny"], 0.0, 1.0, 0.0, 1.0, True)
        kx, ky = (int(k) for k in rng.integers(1, 3, 2))
        u = 0.5 + torch.sin(2 * math.pi * kx * m.x + rng.uniform(0, 6.3)) * torch.cos(2 * math.pi * ky * m.y)
        yield c, op, m, u


def _poisson_data(case, seed):
    """operators, mesh, source f = lap u - shift u and Dirichlet values g [K][3][Nfp] of a smooth random u"""
    rng = np.random.default_rng(seed)
    op = _operators(case["N"])
    m = _Mesh(op, case["nx"], case["ny"], 0.0, 1.0, 0.0, 1.0, False)
    u, lap = torch.zeros_like(m.x), torch.zeros_like(m.x)
    for _ in range(3):
        kx, ky = (math.pi * int(k) for k in rng.integers(1, 5, 2))
        a, px, py = rng.uniform(0.5, 1.0), rng.uniform(0, 2 * math.pi), rng.uniform(0, 2 * math.pi)
        w = a * torch.sin(kx * m.x + px) * torch.sin(ky * m.y + py)
        u, lap = u + w, lap - (kx * kx + ky * ky) * w
    return op, m, lap - case["shift"] * u, u.reshape(-1)[m.own]


def prepare(case, seed):
    from hopefoam_amd import dgh
    ctx = dgh.Context(0)
    s = dict(case=case, ctx=ctx)
    host = lambda t: t.contiguous().cpu().numpy()  # noqa: E731
    N = case.get("N")
    if case["kind"] == "ensemble":
        members = list(_ensemble_states(case, seed))
        s["ens"] = ctx.ensemble([m[0] for m in members], autotune=True)
        s["u0"] = [host(m[3]) for m in members]
    elif case["kind"] == "poisson":
        _, _, f, g = _poisson_data(case, seed)
        mesh = ctx.mesh_structured(N, case["nx"], case["ny"], 0.0, 1.0, 0.0, 1.0, periodic=(False, False),
                                   bc_tag=dgh.DGH_BC_FIXED_VALUE)
        s["solver"] = mesh.sipg(penalty=dgh.DGH_SIPG_PENALTY_H if case["penalty"] == "h" else
                                dgh.DGH_SIPG_PENALTY_REFERENCE,
                                pc=dgh.DGH_PC_BLOCK_JACOBI if case["pc"] == "block" else dgh.DGH_PC_JACOBI,
                                mode=dgh.DGH_SOLVE_MIXED if case["mode"] == "mixed" else dgh.DGH_SOLVE_FP64,
                                # the projection solver's tolerance; the benchmark's for the mixed solver
                                rtol=1e-10 if case["mode"] == "mixed" else 1e-12, maxit=200000,
                                mass_shift=case["shift"])
        s["f_host"], s["g"] = host(f), host(g)
        s["f"], s["b"], s["u"], s["zero"] = mesh.field(1), mesh.field(1), mesh.field(1), mesh.field(1)
    else:
        _, _, q, p = _flow(case, seed)
        bc = {"periodic": dgh.DGH_BC_DEFAULT, "open": dgh.DGH_BC_ZERO_GRADIENT, "inflow": dgh.DGH_BC_FIXED_VALUE}
        per = case["bc"] == "periodic"
        mesh = ctx.mesh_structured(N, case["nx"], case["ny"], *_box(case), periodic=(per, per), bc_tag=bc[case["bc"]])
        s["mesh"], s["vortex"], s["q_host"] = mesh, p, host(q)
        nvar = q.shape[0]
        s["q"] = mesh.field(nvar)
        if case["kind"] != "limit":
            flux = {"upwind": dgh.DGH_FLUX_UPWIND, "lf": dgh.DGH_FLUX_LF, "roe": dgh.DGH_FLUX_ROE}[case["flux"]]
            prec = {"fp64": dgh.DGH_PREC_FP64, "fp32": dgh.DGH_PREC_FP32, "bf16x3": dgh.DGH_PREC_BF16X3}[case["prec"]]
            s["desc"] = dgh.RhsDesc(dgh.DGH_EQ_ADVECT if nvar == 1 else dgh.DGH_EQ_EULER, flux, prec, 0, 1.0, 1.0,
                                    GAMMA)
        if case["kind"] == "evaluate":
            s["out"] = mesh.field(nvar)
        if case["kind"] == "run":
            s["q0"] = mesh.field(nvar, s["q_host"])
            s["dt"] = _time_step(case, q)
            s["limiter"] = None
            if case["limiter"] == "mlp":
                from hopefoam_amd.indicator import load_net
                s["net"] = load_net(ctx, os.path.join(ROOT, "hopefoam_amd", "data", "indicator_N%d.npz" % N))
                s["limiter"] = mesh.limiter_desc(M=50.0, mlp=s["net"], threshold=0.5)
            elif case["limiter"] == "tvb":
                s["limiter"] = mesh.limiter_desc(M=50.0, positivity=True)
            elif case["limiter"] == "triangle":
                s["limiter"] = mesh.limiter_desc(kind=dgh.DGH_LIM_TRIANGLE, positivity=True, eps=1e-2)
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "ensemble":
        for i, u in enumerate(s["u0"]):
            s["ens"].set(i, u)
        s["ens"].run(case["steps"], graph=True)
        return [np.concatenate([s["ens"].get(i).reshape(-1) for i in range(len(s["u0"]))])]
    if case["kind"] == "poisson":
        s["f"].upload(s["f_host"])
        s["solver"].rhs(s["f"], s["b"], s["g"])
        s["u"].copy_from(s["zero"])
        s["solver"].solve(s["b"], s["u"])
        return [s["u"].download()]
    if case["kind"] == "evaluate":
        s["q"].upload(s["q_host"])
        s["mesh"].rhs(s["desc"], s["q"], s["out"])
        return [s["out"].download()]
    if case["kind"] == "limit":
        s["q"].upload(s["q_host"])
        if case["limiter"] == "triangle":
            flags, n = s["mesh"].triangle_limit(s["q"])
        else:
            flags, n = s["mesh"].limit(s["q"], M=50.0, positivity=True)
        return [s["q"].download(), flags, n]
    s["q"].copy_from(s["q0"])
    if case["bc"] == "inflow":   # the boundary function restarts the mesh's time as well
        p = s["vortex"]
        s["mesh"].set_bc_function(1, t=0.0, gamma=GAMMA, x0=p[0], y0=p[1], beta=p[2])
    step = s["mesh"].lserk4_run if case["scheme"] == "lserk4" else s["mesh"].ssprk2_run
    step(s["desc"], s["q"], case["steps"], s["dt"], limiter=s["limiter"])
    return [s["q"].download()]


def _stage_work(case, K):
    """bytes and matrix flops of one right-hand side with its stage update: q and the residual in and out, 14
    geometry values and the connectivity; interpolation, two projections and the lift"""
    N, nvar = case["N"], _case_nvar(case)
    Np = (N + 1) * (N + 2) // 2
    wg = 8 if case.get("prec") == "fp64" else 4
    return (K * (Np * nvar * 32 + 14 * wg + 15), K * nvar * (6 * NQ[N] * Np + 6 * Np * (N + 2)))


def work(case):
    if case["kind"] == "ensemble":   # both passes of every stage; the state to the device and back
        b = f = 0
        for c in _ensemble_cases(case):
            K, Np = 2 * c["nx"] * c["ny"], (c["N"] + 1) * (c["N"] + 2) // 2
            stages = 5 * case["steps"]
            b += K * (stages * (72 * Np + 256) + 32 * Np)
            f += K * stages * (8 * Np * Np + 18 * Np * (c["N"] + 1))
        return {"bytes": b, "flops": f}
    N = case["N"]
    K, Np = 2 * case["nx"] * case["ny"], (N + 1) * (N + 2) // 2
    if case["kind"] == "poisson":
        # the source in, the solution out and one operator application, times a floor on the iterations of
        # conjugate gradients on this mesh (they grow with N^2 over the element size, less with a mass shift)
        h = 1.0 / max(case["nx"], case["ny"])
        k2 = 1.0 / (2 * math.pi ** 2 + case["shift"])
        its = max(5.0, 0.5 * (N + 1) ** 2 / h * math.sqrt(k2))
        return {"bytes": K * Np * 8 * (2 + 9 * its), "flops": K * its * (6 * Np * Np + 36 * Np * (N + 2))}
    nvar = _case_nvar(case)
    state = K * Np * nvar * 8
    if case["kind"] == "limit":
        return {"bytes": 6 * state, "flops": 10 * K * Np * nvar}
    b, f = _stage_work(case, K)
    if case["kind"] == "evaluate":
        return {"bytes": 6 * state, "flops": f}
    stages = case["steps"] * (5 if case["scheme"] == "lserk4" else 2)
    if case["limiter"] != "none":
        b += 2 * state
    return {"bytes": stages * b + 4 * state, "flops": stages * f}


# ---------------------------------------------------------------- the same results in 64 bits
def _euler_flux(q):
    p = (GAMMA - 1) * (q[3] - 0.5 * (q[1] ** 2 + q[2] ** 2) / q[0])
    u, v = q[1] / q[0], q[2] / q[0]
    return (torch.stack([q[1], q[1] * u + p, q[1] * v, (q[3] + p) * u]),
            torch.stack([q[2], q[2] * u, q[2] * v + p, (q[3] + p) * v]), p)


def _face_flux(flux, M, P, nx, ny):
    """normal flux of the traces [vars][K][3][g], own M and other P"""
    if flux == "upwind":
        vn = nx + ny
        return 0.5 * (vn * (M + P) + vn.abs() * (M - P))
    (FM, GM, pM), (FP, GP, pP) = _euler_flux(M), _euler_flux(P)
    mean = 0.5 * (nx * (FM + FP) + ny * (GM + GP))
    if flux == "lf":
        lam = torch.maximum(*(((nx * q[1] + ny * q[2]) / q[0]).abs() + torch.sqrt((GAMMA * p / q[0]).abs())
                              for q, p in ((M, pM), (P, pP))))
        return mean + 0.5 * lam * (M - P)
    # Roe's linearisation in the face frame, no entropy fix
    wM, wP = torch.sqrt(M[0]), torch.sqrt(P[0])
    avg = lambda a, b: (wM * a + wP * b) / (wM + wP)  # noqa: E731
    un = [(nx * q[1] + ny * q[2]) / q[0] for q in (M, P)]
    ut = [(nx * q[2] - ny * q[1]) / q[0] for q in (M, P)]
    rho, u, v = wM * wP, avg(*un), avg(*ut)
    H = avg((M[3] + pM) / M[0], (P[3] + pP) / P[0])
    c2 = (GAMMA - 1) * (H - 0.5 * (u * u + v * v))
    c = torch.sqrt(c2.abs())
    dr, du, dv, dp = P[0] - M[0], un[1] - un[0], ut[1] - ut[0], pP - pM
    a1 = 0.5 * (dp / c2 - rho * du / c) * (u - c).abs()
    a2 = (dr - dp / c2) * u.abs()
    a3 = rho * dv * u.abs()
    a4 = 0.5 * (dp / c2 + rho * du / c) * (u + c).abs()
    d0, dn = a1 + a2 + a4, a1 * (u - c) + a2 * u + a4 * (u + c)
    dt = (a1 + a2 + a4) * v + a3
    de = a1 * (H - u * c) + a2 * 0.5 * (u * u + v * v) + a3 * v + a4 * (H + u * c)
    return mean - 0.5 * torch.stack([d0, nx * dn - ny * dt, ny * dn + nx * dt, de])


def _rhs(case, op, m, q, ghost=None):
    nvar, K, Np = q.shape
    flat = q.reshape(nvar, -1)
    qc = q @ op["Vq"].T
    F, G = (qc, qc) if nvar == 1 else _euler_flux(qc)[:2]
    c = lambda a: a[None, :, None]  # noqa: E731
    out = (c(m.rx) * F + c(m.ry) * G) @ op["Pr"].T + (c(m.sx) * F + c(m.sy) * G) @ op["Ps"].T
    other = flat[:, m.other]
    if ghost is not None:
        other = torch.where(m.inner[None, :, :, None], other, ghost)
    M, P = flat[:, m.own] @ op["Vf"].T, other @ op["Vf"].T
    Fn = _face_flux(case["flux"], M, P, m.nx[:, :, None], m.ny[:, :, None])
    return out - (m.fs[None, :, :, None] * Fn).reshape(nvar, K, -1) @ op["lift"].T


def _ldg(op, m, u, c):
    """right-hand side of u_t + div(a u) = nu div(grad u), alternating fluxes, penalty factor 1"""
    bx, by = 1.0, 1.0 / math.pi
    flat = u.reshape(-1)
    side = bx * m.nx + by * m.ny
    side = torch.where(side == 0.0, torch.where(torch.arange(m.K, device=u.device)[:, None] < m.nb, 1.0, -1.0).double(),
                       side)[:, :, None] > 0
    nx, ny, fs = m.nx[:, :, None], m.ny[:, :, None], m.fs[:, :, None]
    um, up = flat[m.own], flat[m.other]
    d = torch.where(side, torch.zeros_like(um), um - up)
    ur, us = u @ op["Dr"].T, u @ op["Ds"].T
    lift = lambda g: g.reshape(m.K, -1) @ op["liftn"].T  # noqa: E731
    e = lambda a: a[:, None]  # noqa: E731
    qx = e(m.rx) * ur + e(m.sx) * us - lift(fs * nx * d)
    qy = e(m.ry) * ur + e(m.sy) * us - lift(fs * ny * d)
    Fx, Fy = c["ax"] * u - c["nu"] * qx, c["ay"] * u - c["nu"] * qy
    div = (e(m.rx) * Fx + e(m.ry) * Fy) @ op["Dr"].T + (e(m.sx) * Fx + e(m.sy) * Fy) @ op["Ds"].T
    fx, fy = qx.reshape(-1), qy.reshape(-1)
    qm, qp = nx * fx[m.own] + ny * fy[m.own], nx * fx[m.other] + ny * fy[m.other]
    an = c["ax"] * nx + c["ay"] * ny
    qh = torch.where(side, qp, qm) - m.fsmax[:, :, None] * (um - up)
    return -div + lift(fs * ((an * um - c["nu"] * qm) - (torch.where(an >= 0, an * um, an * up) - c["nu"] * qh)))


def _lserk4(rhs, q, steps, dt):
    res = torch.zeros_like(q)
    for _ in range(steps):
        for a, b in zip(LSERK_A, LSERK_B):
            res = a * res + dt * rhs(q)
            q = q + b * res
    return q


def _sipg(case, op, m, f, g):
    """solution of the SIPG system by conjugate gradients to round-off"""
    N, K = case["N"], m.K
    Np = op["r"].numel()
    tau = m.fsmax * (N + 1) ** 2 * (1.0 if case["penalty"] == "h" else 20.0)
    e = torch.arange(K, device=f.device)[:, None]
    nbc = m.nb.clamp(min=0)
    # the smaller element of a face owns it and gives the edge length
    js = torch.where(m.inner & (m.nb < e), m.Js[nbc, m.nf], m.Js)
    w = js[:, :, None] * op["gw"]
    ar = m.nx * m.rx[:, None] + m.ny * m.ry[:, None]
    as_ = m.nx * m.sx[:, None] + m.ny * m.sy[:, None]
    c1, c2, c3 = (m.J * v for v in (m.rx ** 2 + m.ry ** 2, m.rx * m.sx + m.ry * m.sy, m.sx ** 2 + m.sy ** 2))
    k = lambda a: a[:, None]  # noqa: E731
    Srs = op["Srs"] + op["Srs"].T
    fr, inner = op["fm"], m.inner[:, :, None]
    VfD = [[op["Vf"] @ op[D][fr[f]] for f in range(3)] for D in ("Dr", "Ds")]

    def normal(u):   # own n . grad at the face Gauss points
        return torch.stack([ar[:, f, None] * (u @ VfD[0][f].T) + as_[:, f, None] * (u @ VfD[1][f].T)
                            for f in range(3)], 1)

    def lifted(av, cv):
        out = torch.zeros(K, Np, dtype=f.dtype, device=f.device)
        for j in range(3):
            out.index_add_(1, fr[j], av[:, j] @ op["Vf"])
            out += (ar[:, j, None] * cv[:, j]) @ VfD[0][j] + (as_[:, j, None] * cv[:, j]) @ VfD[1][j]
        return out

    def S(u):        # minus the reference's (negative) operator, mass shift included
        ue = u.reshape(-1)[m.own] @ op["Vf"].T
        un = u.reshape(-1)[m.other] @ op["Vf"].T
        dn = normal(u)
        dnn = -dn[nbc, m.nf].flip(2)
        t = tau[:, :, None]
        av = torch.where(inner, w * (-0.5 * t * (ue - un) + 0.5 * (dn + dnn)), w * (-t * ue + dn))
        cv = torch.where(inner, 0.5 * w * (ue - un), w * ue)
        vol = k(c1) * (u @ op["Srr"]) + k(c2) * (u @ Srs) + k(c3) * (u @ op["Sss"])
        return vol - lifted(av, cv) + case["shift"] * k(m.J) * (u @ op["M"])

    gq = torch.where(inner, torch.zeros_like(w), g @ op["Vf"].T)
    rhs = -(k(m.J) * (f @ op["M"]) + lifted(-w * tau[:, :, None] * gq, w * gq))
    # element blocks of S as the preconditioner: the couplings inside one element
    dia = torch.zeros(K, Np, Np, dtype=f.dtype, device=f.device)
    dia += c1[:, None, None] * op["Srr"] + c2[:, None, None] * Srs + c3[:, None, None] * op["Sss"]
    dia += case["shift"] * m.J[:, None, None] * op["M"]
    for j in range(3):
        V = torch.zeros(N + 2, Np, dtype=f.dtype, device=f.device)
        V[:, fr[j]] = op["Vf"]
        half = torch.where(m.inner[:, j], 0.5, 1.0).double()
        wj = w[:, j] * half[:, None]
        cross = lambda A: torch.einsum("ge,kg,gf->kef", V, wj, A)  # noqa: E731
        dia += tau[:, j, None, None] * cross(V)
        for a, D in ((ar, VfD[0][j]), (as_, VfD[1][j])):
            x = a[:, j, None, None] * cross(D)
            dia -= x + x.transpose(1, 2)
    inv = torch.linalg.inv(dia)
    B = lambda r: (inv * r[:, None, :]).sum(2)  # noqa: E731
    u = torch.zeros_like(rhs)
    for _ in range(3):   # restarts from the true residual take off what the recurrence lost
        r = rhs - S(u)
        z = B(r)
        p, rz = z, (r * z).sum()
        stop = 1e-13 * (B(rhs) * rhs).sum().sqrt()
        for it in range(20000):
            if it % 50 == 0 and float(rz.clamp(min=0).sqrt()) <= float(stop):
                break
            Sp = S(p)
            a = rz / (p * Sp).sum()
            u, r = u + a * p, r - a * Sp
            z = B(r)
            new = (r * z).sum()
            p, rz = z + new / rz * p, new
    return u


def exact(case, seed):
    host = lambda t: t.cpu().numpy()  # noqa: E731
    if case["kind"] == "ensemble":
        out = [_lserk4(lambda v: _ldg(op, m, v, c), u, case["steps"], c["dt"]).reshape(-1)
               for c, op, m, u in _ensemble_states(case, seed)]
        return [host(torch.cat(out))]
    if case["kind"] == "poisson":
        op, m, f, g = _poisson_data(case, seed)
        return [host(_sipg(case, op, m, f, g))]
    if case["kind"] == "limit" or case.get("limiter") in ("tvb", "triangle"):
        return None   # limited states: selected cell by cell by the limiter's own decisions
    # (the learned indicator flags no cell of the smooth vortex: its run is the unlimited one)
    op, m, q, p = _flow(case, seed)
    shape = q.shape if q.shape[0] > 1 else q.shape[1:]
    if case["kind"] == "evaluate":
        return [host(_rhs(case, op, m, q).reshape(shape))]
    dt = _time_step(case, q)
    if case["scheme"] == "lserk4":
        return [host(_lserk4(lambda v: _rhs(case, op, m, v), q, case["steps"], dt).reshape(shape))]
    ghost, x, y = None, m.x.reshape(-1)[m.own], m.y.reshape(-1)[m.own]
    for k in range(case["steps"]):
        if case["bc"] == "inflow":   # both stages see the boundary values of the step's start
            ghost = _vortex(x, y, p, k * dt)
        q1 = q + dt * _rhs(case, op, m, q, ghost)
        q = 0.5 * (q + q1 + dt * _rhs(case, op, m, q1, ghost))
    return [host(q.reshape(shape))]
