"""Performance cases of the operator-apply-and-solve path.

Each case is one call, or one short sequence of calls, that a program using
the package makes: an operator apply, the element operators composed as
opLHS composes them, the convective term and its transpose, the solvers, the
steady adjoint gradient, and the convection-diffusion time loop with its
gradient. Meshes are the deformed sin-sin mesh of the benchmark; random fields
are drawn per global node, so they are continuous.

  listed()              the named cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   mesh, operator, plan and inputs on the GPU
  run(state)            one pass
  work(case)            bytes and operations a pass cannot do without
  exact(case, seed)     run's outputs in plain torch, in 64 bits
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "spectralelements.jl_amd"))

import semhip as se  # noqa: E402
from semhip import workloads  # noqa: E402

AMP = 0.1          # deformation amplitude of the benchmark mesh
DT = 1e-3          # time step and diffusivity of the cd2d problem
NU_CD = 1e-3


def listed():
    return [
        # The smallest call: one Poisson apply on the 4x4-element, N = 8 mesh of
        # the manufactured-solution problem. Launches and host time.
        {"name": "apply_4x4_p9", "kind": "apply", "nr": 9, "ns": 9, "Ex": 4, "Ey": 4,
         "per": 0, "k": 0.0, "prec": "f64"},
        # The headline apply: Helmholtz, 256x256 elements, N = 7, FP64.
        {"name": "apply_256x256_p8", "kind": "apply", "nr": 8, "ns": 8, "Ex": 256, "Ey": 256,
         "per": 0, "k": 1.0, "prec": "f64"},
        # opLHS as the equations compose it, hlmz with a viscosity field, then
        # gatherScatter, then mask, on a ragged mesh that is periodic in x.
        {"name": "ops_83x57_p11_periodic", "kind": "ops", "nr": 11, "ns": 11, "Ex": 83, "Ey": 57,
         "per": 1, "k": 1.0, "prec": "f64"},
        # The dealiased convective term and its transpose (one explicit term of
        # a time step and of its adjoint), N = 7 with 12 dealiasing points.
        {"name": "advect_96x96_p8_pd12", "kind": "advect", "nr": 8, "ns": 8, "pd": 12, "Ex": 96,
         "Ey": 96, "per": 0},
        # The smallest solve: the manufactured-solution Poisson problem, Jacobi.
        {"name": "pcg_4x4_p9", "kind": "pcg", "nr": 9, "ns": 9, "Ex": 4, "Ey": 4, "per": 0,
         "k": 0.0, "prec": "f64"},
        # A Jacobi solve at production size, 128x128 elements, N = 7.
        {"name": "pcg_128x128_p8", "kind": "pcg", "nr": 8, "ns": 8, "Ex": 128, "Ey": 128,
         "per": 0, "k": 1.0, "prec": "f64"},
        # A solve on a mesh of different orders in the two directions.
        {"name": "pcg_20x14_nr12_ns9", "kind": "pcg", "nr": 12, "ns": 9, "Ex": 20, "Ey": 14,
         "per": 0, "k": 1.0, "prec": "f64"},
        # The headline solve with the multigrid preconditioner.
        {"name": "mg_256x256_p8", "kind": "mg", "nr": 8, "ns": 8, "Ex": 256, "Ey": 256,
         "per": 0, "k": 1.0, "prec": "f64"},
        # The mixed-precision solve at N = 15: FP32 inner iterations inside FP64
        # residual replacement.
        {"name": "mixed_64x64_p16_f32", "kind": "mixed", "nr": 16, "ns": 16, "Ex": 64, "Ey": 64,
         "per": 0, "k": 1.0, "prec": "f32"},
        # The steady adjoint: forward solve, objective, adjoint solve and the
        # gradient with respect to the variable coefficient.
        {"name": "adjoint_64x64_p8", "kind": "adjoint", "nr": 8, "ns": 8, "Ex": 64, "Ey": 64,
         "per": 0},
        # The cd2d forecast: BDF2/EXT2 steps from a Gaussian blob, N = 9.
        {"name": "cd_64x64_p10_20steps", "kind": "cd", "nr": 10, "ns": 10, "pd": 15, "Ex": 64,
         "Ey": 64, "per": 0, "steps": 20},
        # The gradient of the time-integrated objective through the loop, with
        # checkpointing.
        {"name": "cdgrad_32x32_p8_12steps", "kind": "cdgrad", "nr": 8, "ns": 8, "pd": 12,
         "Ex": 32, "Ey": 32, "per": 0, "steps": 12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _elements(rng, nr, ns, lo, hi, nmax):
    """Element counts spread over their logarithm, with at most nmax nodes."""
    while True:
        Ex, Ey = _log_int(rng, lo, hi), _log_int(rng, lo, hi)
        if nr * ns * Ex * Ey <= nmax:
            return Ex, Ey


def draw(rng):
    kind = rng.choice(["apply", "ops", "advect", "pcg", "pcg", "mg", "mixed", "adjoint", "cd",
                       "cdgrad"])
    c = {"kind": kind, "per": 0}
    if kind == "apply":
        p = rng.randint(4, 16)
        c.update(nr=p, ns=p, k=rng.choice([0.0, 1.0]), prec=rng.choice(["f64", "f64", "f32"]),
                 per=rng.choice([0, 0, 1]))
        c["Ex"], c["Ey"] = _elements(rng, p, p, 4, 300, 1 << 22)
    elif kind == "ops":
        nr = rng.randint(4, 18)
        ns = nr if rng.random() < 0.5 else rng.randint(4, 18)
        c.update(nr=nr, ns=ns, k=1.0, prec="f64", per=rng.choice([0, 1]))
        c["Ex"], c["Ey"] = _elements(rng, nr, ns, 4, 160, 1 << 20)
    elif kind == "advect":
        p = rng.randint(4, 12)
        c.update(nr=p, ns=p, pd=(3 * p + 1) // 2)
        c["Ex"], c["Ey"] = _elements(rng, p, p, 6, 110, 600000)
    elif kind == "pcg":
        if rng.random() < 0.3:
            nr, ns = rng.randint(5, 14), rng.randint(5, 14)
            c.update(nr=nr, ns=ns)
            c["Ex"], c["Ey"] = _elements(rng, nr, ns, 4, 24, 30000)
        else:
            p = rng.randint(4, 12)
            c.update(nr=p, ns=p)
            c["Ex"], c["Ey"] = _elements(rng, p, p, 4, min(128, 1024 // p), 1 << 20)
        c.update(k=rng.choice([0.0, 1.0]), prec="f64")
    elif kind == "mg":
        p = rng.choice([4, 5, 8, 8, 12, 16])
        c.update(nr=p, ns=p, k=rng.choice([0.0, 1.0]), prec=rng.choice(["f64", "f64", "f32"]))
        q = rng.choice([1, 2, 4, 8])
        Ex, Ey = _elements(rng, p, p, 8, 256, 1 << 21)
        c["Ex"], c["Ey"] = max(q, Ex // q * q), max(q, Ey // q * q)
    elif kind == "mixed":
        c.update(nr=16, ns=16, k=1.0, prec=rng.choice(["f32", "f32", "f16x3"]))
        c["Ex"], c["Ey"] = rng.randint(12, 52), rng.randint(12, 52)
    elif kind == "adjoint":
        p = rng.randint(4, 9)
        c.update(nr=p, ns=p)
        c["Ex"], c["Ey"] = _elements(rng, p, p, 6, 60, 200000)
    else:
        p = rng.randint(5, 10)
        c.update(nr=p, ns=p, pd=(3 * p + 1) // 2)
        if kind == "cd":
            c["steps"] = rng.randint(6, 20)
            c["Ex"], c["Ey"] = _elements(rng, p, p, 8, 64, 400000)
        else:
            c["steps"] = rng.randint(4, 12)
            c["Ex"], c["Ey"] = _elements(rng, p, p, 6, 36, 65000)
    return c


# ------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _local_index(n, E, per):
    """Global index of each local row of E elements of n points."""
    i = torch.arange(E, device="cuda").reshape(E, 1) * (n - 1) + torch.arange(n, device="cuda")
    i = i.reshape(-1)
    return i % (E * (n - 1)) if per else i


def _normal(case, gen):
    """N(0, 1) per global node, on the local copies."""
    gx = _local_index(case["nr"], case["Ex"], case["per"])
    gy = _local_index(case["ns"], case["Ey"], 0)
    g = torch.randn(int(gx.max()) + 1, int(gy.max()) + 1, generator=gen, device="cuda",
                    dtype=torch.float64)
    return g[gx][:, gy]


def _inputs(case, seed):
    """The random inputs of a case; the same on the package's and the plain side."""
    gen = _gen(seed)
    kind = case["kind"]
    if kind in ("apply", "pcg", "mg", "mixed"):
        return {"f": _normal(case, gen)}
    if kind in ("ops", "advect"):
        return {"f": _normal(case, gen), "w": _normal(case, gen)}
    rng = np.random.default_rng(seed)
    if kind == "adjoint":
        return {"nu_seed": int(rng.integers(1 << 30)), "us_seed": int(rng.integers(1 << 30))}
    return {"x0": float(rng.uniform(0.3, 0.6)), "y0": float(rng.uniform(-0.2, 0.2))}


def _mesh(case, n=None):
    return se.Mesh(n or case["nr"], n or case["ns"], case["Ex"], case["Ey"],
                   (bool(case["per"]), False), se.deform_sinsin(AMP))


def _tol(case, b):
    # relative to the right-hand side: the tolerances of the adjoint and time
    # stepping solvers (1e-12), of the headline solve (1e-10, which multigrid
    # overshoots), and one at which the mixed solve's own error is small
    return {"mg": 1e-10, "mixed": 1e-11}.get(case["kind"], 1e-12) * float(b.abs().max())


# --------------------------------------------------------------- the package
def prepare(case, seed):
    v = _inputs(case, seed)
    kind = case["kind"]
    m = _mesh(case)
    M = se.generateMask("DDDD", m)
    s = {"kind": kind, "m": m, "M": M}
    if kind == "apply":
        s["op"] = se.SEMOperator(1.0, case["k"], m, M, precision=case["prec"])
        s["u"] = se.to_device(v["f"], dtype=s["op"].dtype)
    elif kind == "ops":
        s["u"] = se.to_device(v["f"])
        s["nu"] = se.to_device(1.0 + 0.5 * torch.tanh(v["w"]))
        s["k"] = case["k"]
    elif kind == "advect":
        s["mD"] = _mesh(case, case["pd"])
        s["T"], s["w"] = se.to_device(v["f"]), se.to_device(v["w"])
        s["vx"], s["vy"] = se.to_device(-m.y), se.to_device(m.x)
    elif kind in ("pcg", "mg", "mixed"):
        s["op"] = se.SEMOperator(1.0, case["k"], m, M)
        s["b"] = se.gatherScatter(se.mask(se.mass(se.to_device(v["f"]), m), M), m)
        s["tol"] = _tol(case, s["b"])
        s["mult"] = m.mult
        if kind == "mg":
            s["opM"] = se.MG(s["op"], precision=case["prec"])
        else:
            s["d"] = s["op"].jacobi()
        if kind == "mixed":
            s["op_lo"] = se.SEMOperator(1.0, case["k"], m, M, precision=case["prec"])
        elif kind == "pcg":
            s["opM"] = se.Diagonal(s["d"])
    elif kind == "adjoint":
        s["nu"] = workloads.coefficient_field(m, v["nu_seed"]).requires_grad_(True)
        s["us"] = 0.1 * workloads.coefficient_field(m, v["us_seed"])
        s["B"] = m.B
        s["problem"] = se.VarDiffusion(m, M, torch.ones_like(s["us"]))
        s["solver"] = se.diffusion_solver()
    else:
        mD = _mesh(case, case["pd"])
        fld = se.Field("DDDD", m, 2)
        s["cdn"] = se.ConvectionDiffusion("cd2d", fld, -m.y, m.x,
                                          se.TimeStepper(0.0, case["steps"] * DT, DT, 2), mD,
                                          nu=NU_CD)
        s["u0"] = workloads.gaussian_blob(m, v["x0"], v["y0"])
        s["steps"] = case["steps"]
    return s


def run(s):
    kind = s["kind"]
    if kind == "apply":
        return s["op"](s["u"])
    if kind == "ops":
        return se.mask(se.gatherScatter(se.hlmz(s["u"], s["nu"], s["k"], s["m"]), s["m"]), s["M"])
    if kind == "advect":
        return (se.advect(s["T"], s["vx"], s["vy"], s["m"], s["mD"]),
                se.advect(s["w"], s["vx"], s["vy"], s["m"], s["mD"], transpose=True))
    if kind in ("pcg", "mg"):
        return se.pcg(s["b"], s["op"], opM=s["opM"], mult=s["mult"], tol=s["tol"])
    if kind == "mixed":
        return se.pcg_mixed(s["b"], s["op"], s["op_lo"], d=s["d"], tol=s["tol"])
    if kind == "adjoint":
        u = se.linsolve(s["nu"], s["problem"], s["solver"])
        J = 0.5 * torch.sum(s["B"] * (u - s["us"]) ** 2)
        (g,) = torch.autograd.grad(J, s["nu"])
        return {"u": u.detach(), "J": J.detach(), "grad": g}
    if kind == "cd":
        s["cdn"].reset_(s["u0"])
        s["cdn"].run_(s["steps"])
        return s["cdn"].fld.u
    r = se.cd_gradient(s["cdn"], s["u0"], s["steps"])
    return {"J": r.J, "grad": r.grad}


# --------------------------------------------------------------------- work
def work(case):
    """One read of every input field and factor and one write of every output
    per apply; a solve's iterations (estimated: a Jacobi solve takes about
    six per node row of the longer side, a solve of a time step 25, a
    multigrid solve 12 of about 12 fine-level applies each) repeat the
    operations, and the bytes of a solve are those of one iteration, its
    fields read once."""
    nr, ns = case["nr"], case["ns"]
    n = nr * ns * case["Ex"] * case["Ey"]
    kind = case["kind"]
    w = 4 if case.get("prec") == "f32" and kind == "apply" else 8
    app = n * (4 * (nr + ns) + 11)          # one operator apply
    it = app + 14 * n                       # one PCG iteration
    its = 6 * max(nr * case["Ex"], ns * case["Ey"])
    if kind == "apply":
        return {"bytes": n * w * (6 if case["k"] else 5), "flops": app}
    if kind == "ops":
        return {"bytes": n * 8 * 7, "flops": app + 4 * n}
    if kind in ("pcg", "mixed"):
        return {"bytes": n * 8 * (6 + (case["k"] != 0.0)), "flops": its * it}
    if kind == "mg":
        return {"bytes": n * 8 * (5 + (case["k"] != 0.0)), "flops": 12 * 12 * it}
    if kind == "adjoint":
        return {"bytes": n * 8 * 15, "flops": 2 * its * it}
    pd = case["pd"]
    nd = pd * pd * case["Ex"] * case["Ey"]
    adv = n * 4 * nr + 2 * 5 * (n * pd + nd * nr) + 5 * nd
    if kind == "advect":
        return {"bytes": 8 * (2 * 8 * n + 2 * nd), "flops": 2 * adv}
    step = 25 * it + adv + 10 * n
    if kind == "cd":
        return {"bytes": 8 * (12 * n + nd), "flops": case["steps"] * step}
    return {"bytes": 8 * (14 * n + nd), "flops": 3 * case["steps"] * step}


# -------------------------------------------------------------------- exact
def _gll(n):
    """Gauss-Lobatto-Legendre points and weights: Newton on (1 - x^2) P'."""
    leg = np.polynomial.legendre
    P = leg.Legendre.basis(n - 1)
    d1 = P.deriv(1)
    z = np.concatenate([[-1.0], np.sort(d1.roots().real), [1.0]])
    d2 = d1.deriv(1)
    for _ in range(4):
        z[1:-1] -= d1(z[1:-1]) / d2(z[1:-1])
    z = 0.5 * (z - z[::-1])
    return z, 2.0 / (n * (n - 1) * P(z) ** 2)


def _interp(xo, xi):
    """Lagrange interpolation matrix from points xi to xo."""
    J = np.ones((len(xo), len(xi)))
    for j in range(len(xi)):
        for q in range(len(xi)):
            if q != j:
                J[:, j] *= (xo - xi[q]) / (xi[j] - xi[q])
    return J


def _deriv(z):
    n = len(z)
    D = np.zeros((n, n))
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = np.prod([(z[i] - z[q]) / (z[j] - z[q]) for q in range(n)
                                   if q not in (i, j)]) / (z[j] - z[i])
        D[i, i] = -np.sum(D[i])
    return D


class _Plain:
    """The operators in plain torch, 64 bits, on (Ex, nr, Ey, ns) blocks."""

    def __init__(self, case, n=None):
        nr, ns = n or case["nr"], n or case["ns"]
        self.shape = (nr * case["Ex"], ns * case["Ey"])
        self.blk = (case["Ex"], nr, case["Ey"], ns)
        self.per = bool(case["per"])
        zr, wr = _gll(nr)
        zs, ws = _gll(ns)
        self.zr, self.zs = zr, zs
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        self.Dr, self.Ds = dev(_deriv(zr)), dev(_deriv(zs))

        def nodes(E, z):
            h = 2.0 / E
            return (-1.0 + h * np.arange(E)[:, None] + 0.5 * h * (z + 1.0)[None, :]).reshape(-1)
        X, Y = torch.meshgrid(dev(nodes(case["Ex"], zr)), dev(nodes(case["Ey"], zs)),
                              indexing="ij")
        sn = AMP * torch.sin(math.pi * X) * torch.sin(math.pi * Y)
        self.x, self.y = self.b(X + sn), self.b(Y + sn)
        xr, xs = self.dr(self.x), self.ds(self.x)
        yr, ys = self.dr(self.y), self.ds(self.y)
        J = xr * ys - xs * yr
        self.rx, self.ry, self.sx, self.sy = ys / J, -xs / J, -yr / J, xr / J
        self.B = J * (dev(wr).reshape(1, nr, 1, 1) * dev(ws).reshape(1, 1, 1, ns))
        self.G11 = self.B * (self.rx ** 2 + self.ry ** 2)
        self.G12 = self.B * (self.rx * self.sx + self.ry * self.sy)
        self.G22 = self.B * (self.sx ** 2 + self.sy ** 2)
        one = torch.ones_like(self.B)
        self.mult = 1.0 / self.gs(one)
        self.M = one.clone()
        if not self.per:
            self.M[0, 0] = 0.0
            self.M[-1, -1] = 0.0
        self.M[:, :, 0, 0] = 0.0
        self.M[:, :, -1, -1] = 0.0

    def b(self, u):
        return u.reshape(self.blk)

    def f(self, u):
        return u.reshape(self.shape)

    def dr(self, u):
        return torch.einsum("ak,xkyb->xayb", self.Dr, u)

    def ds(self, u):
        return u @ self.Ds.t()

    def drt(self, u):
        return torch.einsum("ka,xkyb->xayb", self.Dr, u)

    def dst(self, u):
        return u @ self.Ds

    def gs(self, u):
        u = u.clone()
        s = u[:-1, -1] + u[1:, 0]
        u[:-1, -1] = s
        u[1:, 0] = s
        if self.per:
            s = u[-1, -1] + u[0, 0]
            u[-1, -1] = s
            u[0, 0] = s
        s = u[:, :, :-1, -1] + u[:, :, 1:, 0]
        u[:, :, :-1, -1] = s
        u[:, :, 1:, 0] = s
        return u

    def hlmz(self, u, nu, k, fac=1.0):
        ur, us = self.dr(u), self.ds(u)
        a = self.drt(fac * (self.G11 * ur + self.G12 * us)) + self.dst(
            fac * (self.G12 * ur + self.G22 * us))
        return nu * a + k * (self.B * u)

    def A(self, u, nu, k, fac=1.0):
        return self.M * self.gs(self.hlmz(u, nu, k, fac))

    def jacobi(self, nu, k, fac=1.0):
        t1 = torch.einsum("ka,xkyb->xayb", self.Dr ** 2, fac * self.G11)
        t3 = torch.einsum("kb,xayk->xayb", self.Ds ** 2, fac * self.G22)
        dd = torch.diagonal(self.Dr).reshape(1, -1, 1, 1) * torch.diagonal(self.Ds)
        return self.M / self.gs(nu * (t1 + t3 + 2.0 * dd * fac * self.G12) + k * self.B)

    def solve(self, b, nu, k, fac=1.0, rtol=1e-14, most=20000):
        """Jacobi PCG until the residual is at rtol or no longer falls."""
        d = self.jacobi(nu, k, fac)
        x, r = torch.zeros_like(b), b.clone()
        z = d * r
        p, t = z.clone(), (r * z * self.mult).sum()
        goal, best, since = rtol * float(b.abs().max()), math.inf, 0
        for it in range(most):
            w = self.A(p, nu, k, fac)
            a = t / (p * w * self.mult).sum()
            x += a * p
            r -= a * w
            z = d * r
            t, tp = (r * z * self.mult).sum(), t
            p = z + (t / tp) * p
            if it % 25 == 24:
                res = float(r.abs().max())
                best, since = (res, 0) if res < 0.9 * best else (best, since + 1)
                if res <= goal or not res > 0.0 or since > 40:
                    break
        return x

    def grad(self, u):
        ur, us = self.dr(u), self.ds(u)
        return self.rx * ur + self.sx * us, self.ry * ur + self.sy * us

    def advect(self, D, T, vx, vy):
        Jr, Js = (torch.from_numpy(_interp(a, c)).cuda() for a, c in ((D.zr, self.zr),
                                                                      (D.zs, self.zs)))
        up = lambda u: torch.einsum("ik,xkyb->xiyb", Jr, u) @ Js.t()  # noqa: E731
        Tx, Ty = self.grad(T)
        c = D.B * (up(vx) * up(Tx) + up(vy) * up(Ty))
        return torch.einsum("ki,xkyb->xiyb", Jr, c) @ Js

    def advect_t(self, D, w, vx, vy):
        """The transpose of advect in T, by differentiating <w, advect(T)>."""
        T = torch.zeros_like(w, requires_grad=True)
        (g,) = torch.autograd.grad((w * self.advect(D, T, vx, vy)).sum(), T)
        return g


def _bdf(n):
    """BDF1/EXT1 on the first step, BDF2/EXT2 after it: (a, b)."""
    return ([1.0], [1.0 / DT, -1.0 / DT]) if n == 1 else (
        [2.0, -1.0], [1.5 / DT, -2.0 / DT, 0.5 / DT])


def _exact_cd(case, v, gradient):
    m, D = _Plain(case), _Plain(case, case["pd"])
    vx, vy = -m.y, m.x
    u = torch.exp(-((m.x - v["x0"]) ** 2 + (m.y - v["y0"]) ** 2) / (2.0 * 0.1 * 0.1))
    us = [u]
    for n in range(1, case["steps"] + 1):
        a, b = _bdf(n)
        rhs = 0.0
        for i, ai in enumerate(a):
            uh = us[n - 1 - i]
            rhs = rhs - b[1 + i] * m.B * uh - ai * m.advect(D, uh, vx, vy)
        us.append(m.solve(m.gs(m.M * rhs), NU_CD, b[0]))
    if not gradient:
        return m.f(us[-1])
    J = sum(0.5 * DT * (m.B * u * u).sum() for u in us[1:])
    acc = [torch.zeros_like(u) for _ in us]
    for n in range(case["steps"], 0, -1):
        a, b = _bdf(n)
        lam = m.solve(m.gs(m.M * (DT * m.B * us[n] + acc[n])), NU_CD, b[0])
        ct = m.advect_t(D, lam, vx, vy)
        for i, ai in enumerate(a):
            acc[n - 1 - i] += -b[1 + i] * m.B * lam - ai * ct
    return {"J": float(J), "grad": m.f(acc[0])}


def exact(case, seed):
    v = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("cd", "cdgrad"):
        return _exact_cd(case, v, kind == "cdgrad")
    m = _Plain(case)
    if kind == "apply":
        # the operator's own input: rounded where the operator takes FP32 fields
        f = v["f"].float().double() if case["prec"] == "f32" else v["f"]
        return m.f(m.A(m.b(f), 1.0, case["k"]))
    if kind == "ops":
        return m.f(m.A(m.b(v["f"]), m.b(1.0 + 0.5 * torch.tanh(v["w"])), case["k"]))
    if kind == "advect":
        D = _Plain(case, case["pd"])
        return (m.f(m.advect(D, m.b(v["f"]), -m.y, m.x)),
                m.f(m.advect_t(D, m.b(v["w"]), -m.y, m.x)))
    if kind in ("pcg", "mg", "mixed"):
        b = m.gs(m.M * (m.B * m.b(v["f"])))
        return m.f(m.solve(b, 1.0, case["k"], rtol=1e-12 if kind == "mg" else 1e-14))

    def field(s):
        # the 16 random-phase modes of the coefficient's definition
        r = np.random.default_rng(s)
        k, th = r.integers(1, 5, size=(16, 2)), r.uniform(0.0, 2.0 * np.pi, size=16)
        phi = sum(0.25 * torch.cos(math.pi * (float(a) * m.x + float(c) * m.y) + float(t))
                  for (a, c), t in zip(k, th))
        return 1.0 + 0.5 * torch.tanh(phi)
    nu, us = field(v["nu_seed"]), 0.1 * field(v["us_seed"])
    u = m.solve(m.gs(m.M * m.B), 1.0, 0.0, fac=nu)
    e = u - us
    lam = m.solve(m.gs(m.M * (m.B * e)), 1.0, 0.0, fac=nu)
    (ux, uy), (lx, ly) = m.grad(u), m.grad(lam)
    return {"u": m.f(u), "J": 0.5 * (m.B * e * e).sum(),
            "grad": m.f(-m.B * (lx * ux + ly * uy))}
