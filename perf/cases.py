"""The work that users of this library give it, as cases to be timed.

A case is one call sequence of the Python driver over the C ABI: an
evaluation of the right-hand side (with or without its vector-Jacobian
product), a run of time steps with the state read back at its end, a
checkpointed gradient, or a run of an ensemble.  listed() holds the sizes
that the repository's configurations, tests and benchmark use; draw() gives
more of the same families over their whole range.

exact() evaluates the same discrete scheme (orthonormal basis on the
reference triangle, the solver's quadrature, single-precision side lengths,
the numerical fluxes, Runge-Kutta forms and time step rule) in plain torch
float64; gradients come from torch's reverse mode.
"""
import ctypes
import functools
import math
from fractions import Fraction

import numpy as np
import torch
import torch.utils.checkpoint

from dgcuda_amd import _lib as L
from dgcuda_amd import autograd as A
from dgcuda_amd import mesh as M
from dgcuda_amd.ensemble import Ensemble
from dgcuda_amd.solver import Solver

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
PHYS = {"adv": L.ADVECTION, "euler": L.EULER, "swe": L.SWE, "tm": L.MAXWELL_TM,
        "te": L.MAXWELL_TE}
INTEG = {"rk4": L.RK4, "rk2": L.RK2MID, "ssp2": L.SSPRK2, "ssp3": L.SSPRK3}
STAGES = {"rk4": 4, "rk2": 2, "ssp2": 2, "ssp3": 3}
FLUX = {"default": L.FLUX_DEFAULT, "llf": L.FLUX_LLF, "roe": L.FLUX_ROE}
NQ = (1, 3, 6, 12, 16, 25)
BASE = dict(kind="steps", physics="euler", p=2, nx=20, ny=27, domain="periodic", integrator="rk4",
            flux="default", limiter=False, cfl=0.0, steps=10)


def _case(name, **kw):
    c = dict(BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a program that brings its own time integrator asks for one right-hand
        # side at a time; on a small mesh (1,080 triangles, the size of the
        # reference's smallest rotating-hill mesh) the call itself is what counts
        _case("rhs_euler_p1_1k", kind="rhs", p=1),
        # the same with its gradient: a torch training step through one
        # evaluation (forward and vector-Jacobian product), ragged mesh
        _case("rhs_vjp_swe_p2_50k", kind="vjp", physics="swe", nx=157, ny=161, domain="walled"),
        # the plain benchmark configuration: advection, 64 x 64 quads, 100 steps
        _case("adv_p1_8k_100", physics="adv", p=1, nx=64, ny=64, integrator="ssp2", cfl=0.3,
              steps=100),
        # the reference's one published timing: the rotating hill at p = 4 on
        # 1,080 triangles, time-dependent inflow on every side
        _case("hill_p4_1k_50", physics="adv", p=4, domain="hill", steps=50),
        # the reference's benchmark sweep: supersonic vortex, walls, inflow
        # and outflow, RK4; its third mesh has 2,880 triangles
        _case("supersonic_p3_3k_25", p=3, nx=16, ny=90, domain="annulus", steps=25),
        # shocks: p = 1 with the slope limiter, the sweep's largest mesh
        _case("limited_p1_12k_20", p=1, nx=32, ny=180, domain="annulus", limiter=True, steps=20),
        # the headline benchmark: isentropic vortex, 524,288 triangles, p = 2
        _case("euler_p2_524k_10", nx=512, ny=512, integrator="ssp3", cfl=0.2, steps=10),
        # a cavity with a permittivity per element, p = 3, RK4
        _case("te_p3_200k_10", physics="te", p=3, nx=316, ny=316, domain="walled", steps=10),
        # its gradient with respect to the initial state and the permittivity
        _case("te_p3_200k_grad_32", kind="adjoint", physics="te", p=3, nx=316, ny=316,
              domain="walled", steps=32, every=16),
        # the largest forward run: p = 4, 2,097,152 triangles
        _case("euler_p4_2m_3", p=4, nx=1024, ny=1024, integrator="ssp3", cfl=0.2, steps=3),
        # a gradient of the total entropy at p = 4
        _case("euler_p4_131k_grad_8", kind="adjoint", p=4, nx=256, ny=256, integrator="ssp3",
              cfl=0.2, steps=8, every=0),
        # many uneven shallow-water meshes and orders stepped together
        _case("ens_swe_roe_16", kind="ensemble", physics="swe", flux="roe", domain="walled",
              integrator="ssp3", p=3, nx=32, ny=200, count=16, steps=20),
    ]


def draw(rng):
    kind = rng.choice(["rhs", "vjp", "steps", "steps", "steps", "adjoint", "ensemble"])
    if kind == "ensemble":  # instances of 2 nx^2 ... 2 ny^2 triangles, orders 1 ... p
        nx = rng.randint(12, 40)
        return _case("", kind=kind, physics="swe", flux=rng.choice(["roe", "llf"]),
                     domain="walled", integrator=rng.choice(["ssp3", "ssp2"]),
                     p=rng.randint(1, 3), nx=nx, ny=rng.randint(60, 180),
                     count=rng.randint(3, 16), steps=rng.randint(5, 20))
    ph = rng.choice(["adv", "euler", "euler", "swe", "tm", "te"])
    c = dict(kind=kind, physics=ph, p=rng.randint(0, 5),
             integrator=rng.choice(["rk4", "ssp3", "ssp2", "rk2"]),
             domain={"adv": ["periodic", "hill"], "euler": ["periodic", "annulus"],
                     "tm": ["periodic", "walled"]}.get(ph, ["walled", "walled"])[rng.randint(0, 1)])
    if ph == "swe":
        c["flux"] = rng.choice(["roe", "llf"])
    if kind == "adjoint":
        # (the entropy of a vortex or the received energy of a pulse)
        c["physics"] = ph = "te" if ph in ("te", "tm", "adv") else "euler"
        c["domain"] = "walled" if ph == "te" else "periodic"
        c["flux"] = "default"
        c["p"] = max(1, c["p"])
        c["every"] = rng.choice([0, 4, 8])
    if kind == "steps" and ph == "euler" and rng.random() < 0.25:
        c.update(p=1, limiter=True)
    nv = L.NVARS[PHYS[ph]]
    n_p = (c["p"] + 1) * (c["p"] + 2) // 2
    kmax = min(524288, int((2.4e6 if kind == "adjoint" else 1.2e7) / (n_p * nv)))
    K = math.exp(rng.uniform(math.log(180), math.log(kmax)))
    nx = max(3, round(math.sqrt(K / 2) * rng.uniform(0.7, 1.0)))
    c.update(nx=nx, ny=max(3, round(K / 2 / nx)), cfl=rng.choice([0.0, 0.2, 0.3]))
    stages = STAGES[c["integrator"]]
    c["steps"] = int(min(rng.randint(8, 60), max(4, 3e9 / (K * n_p * nv * stages * NQ[c["p"]]))))
    if kind == "adjoint":
        c["steps"] = min(c["steps"], 16)
    return _case("", **c)


# ------------------------------------------------------------ setting a case up


@functools.lru_cache(maxsize=24)
def _mesh(domain, nx, ny, seed=20261202):
    """the seeded jittered mesh of a case (a program reads it from a file)"""
    if domain == "periodic1":  # unit square
        return M.structured(nx, ny, periodic=True, jitter=0.2, seed=seed)
    if domain == "periodic10":
        return M.structured(nx, ny, lx=10.0, ly=10.0, periodic=True, jitter=0.2, seed=seed)
    if domain == "hill":
        return M.structured(nx, ny, lx=2.0, ly=2.0, x0=-1.0, y0=-1.0, periodic=False, jitter=0.2,
                            seed=seed, bc=(-3, -3, -3, -3))
    if domain == "annulus":  # x is the radius, y the angle; outflow at angle 0
        m = M.structured(nx, ny, lx=0.384, ly=math.pi / 2, x0=1.0, y0=0.0, periodic=False,
                         jitter=0.1, seed=seed, bc=(-2, -1, -3, -1))
        for a in (m.V, m.side_xy):
            for q in range(0, a.shape[0], 2):
                r, th = a[q].copy(), a[q + 1].copy()
                a[q], a[q + 1] = r * np.cos(th), r * np.sin(th)
        return m
    return M.structured(nx, ny, periodic=False, jitter=0.2, seed=seed, bc=(-1, -1, -1, -1))


def _mesh_of(c):
    d = c["domain"]
    if d == "periodic":
        d = "periodic10" if c["physics"] == "euler" else "periodic1"
    return _mesh(d, c["nx"], c["ny"])


def _problem(c, seed):
    """(problem id, its parameters)"""
    r = np.random.default_rng(seed)
    if c["physics"] == "adv":
        return (L.PROB_ADV_ROTHILL, ()) if c["domain"] == "hill" else (L.PROB_ADV_SINSIN, ())
    if c["physics"] == "euler":
        if c["domain"] == "annulus":
            return L.PROB_EULER_SUPERSONIC, ()
        return L.PROB_EULER_VORTEX, (r.uniform(4, 5), r.uniform(3, 7), r.uniform(3, 7), 1., 1., 10.)
    if c["physics"] == "swe":
        return L.PROB_SWE_BUMP, (1., 0.1, r.uniform(), r.uniform(), r.uniform(0.05, 0.2), 1.)
    return L.PROB_MAXWELL_PULSE, (1., r.uniform(0.3, 0.7), r.uniform(0.3, 0.7), 0.1)


def _solver_args(c, seed):
    prob, prm = _problem(c, seed)
    return dict(integrator=INTEG[c["integrator"]], flux=FLUX[c["flux"]], cfl=c["cfl"], g=9.81,
                problem=prob, problem_params=prm)


def _eps(c, K, seed):
    if c["physics"] != "te":
        return None
    return np.random.default_rng(seed + 17).uniform(1.0, 4.0, K)


def _instances(c, seed):
    """an ensemble's instances as cases of their own (the meshes and orders
    are the case's, the bumps the seed's)"""
    r = np.random.default_rng(7)
    out = []
    for i in range(c["count"]):
        n = round(math.exp(r.uniform(math.log(c["nx"]), math.log(c["ny"]))))
        out.append((dict(c, kind="steps", p=int(r.integers(1, c["p"] + 1)), nx=n, ny=n),
                    seed * 1000 + i))
    return out


def prepare(case, seed):
    c = case
    if c["kind"] == "ensemble":
        inst = _instances(c, seed)
        kw = _solver_args(c, seed)
        E = Ensemble(physics=PHYS[c["physics"]], **kw)
        out = []
        for ci, si in inst:
            E.add(_mesh_of(ci), ci["p"], _problem(ci, si)[1])
        E.build()
        for i, (ci, si) in enumerate(inst):
            u = _initial(ci, si)
            out.append(torch.empty(E.shapes[i], dtype=F64, device=DEV))
            torch.cuda.synchronize()  # the ensemble's stream does not wait for torch's
            _ens_chk(E, E.lib.dg_ens_set_coeffs(E.e, i, L.ptr(u), L.DEVICE))
        torch.cuda.synchronize()
        return dict(case=c, E=E, out=out)
    m = _mesh_of(c)
    s = Solver(PHYS[c["physics"]], c["p"], limiter=c["limiter"], **_solver_args(c, seed))
    s.set_mesh(m)
    eps = _eps(c, m.K, seed)
    if eps is not None:
        s.set_eps(eps)
    u = _initial(c, seed)
    st = dict(case=c, s=s, u=u, out=torch.empty(s.shape, dtype=F64, device=DEV))
    torch.cuda.synchronize()  # the solver's stream does not wait for torch's
    if c["kind"] == "steps":
        s.set_coeffs(u)
    elif c["kind"] == "vjp":
        st["u"] = u.requires_grad_(True)
        st["g"] = _weights(c, seed, s.shape)
    elif c["kind"] == "adjoint":
        st["u"] = u.requires_grad_(True)
        st["dt"] = _adjoint_dt(c, seed, u.detach())
        if eps is not None:
            st["eps"] = torch.tensor(eps, device=DEV, requires_grad=True)
            s.set_objective(L.OBJ_PATCH_SQ, PATCH)
        else:
            s.set_objective(L.OBJ_ENTROPY)
    torch.cuda.synchronize()
    return st


PATCH = (0.45, 0.55, 0.3, 0.4, 2)


def _weights(c, seed, shape):
    g = torch.Generator(device="cpu").manual_seed(seed + 3)
    return torch.randn(shape, generator=g, dtype=F64).to(DEV)


def _ens_chk(E, rc):
    if rc != 0:
        raise L.DgError(rc, (E.lib.dg_ens_last_error(E.e) or b"").decode())


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "rhs":
        return state["s"].eval_rhs(state["u"], t=0.0, dt=0.01, out=state["out"])
    if kind == "vjp":
        k = A.rhs(state["s"], state["u"], t=0.0, dt=0.01)
        (gu,) = torch.autograd.grad(k, state["u"], state["g"])
        return {"k": k.detach(), "gu": gu}
    if kind == "steps":
        # the run goes on from where the last pass left it
        t, _ = state["s"].step(c["steps"], t=state.get("t", 0.0))
        state["t"] = t
        return {"c": state["s"].coeffs(out=state["out"]), "t": t}
    if kind == "adjoint":
        eps = state.get("eps")
        J = A.objective(state["s"], state["u"], c["steps"], state["dt"], eps=eps, every=c["every"])
        g = torch.autograd.grad(J, [state["u"]] + ([eps] if eps is not None else []))
        return {"J": J.detach(), "g": list(g)}
    E = state["E"]
    E.step(c["steps"])
    for i, o in enumerate(state["out"]):
        _ens_chk(E, E.lib.dg_ens_get_coeffs(E.e, i, ctypes.c_void_p(o.data_ptr()), L.DEVICE))
    return state["out"]


def work(case):
    """bytes: per stage the state read, its successor written, the step base
    where the scheme needs it, the metric (52 B an element, 40 B a side);
    flops: interpolation, projection and fluxes of every point."""
    c = case
    if c["kind"] == "ensemble":
        w = [work(ci) for ci, _ in _instances(c, 0)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    K, N, p = 2 * c["nx"] * c["ny"], L.NVARS[PHYS[c["physics"]]], c["p"]
    n_p = (p + 1) * (p + 2) // 2
    mesh, D = 52 * K + 60 * K, 8 * K * n_p * N
    ops = K * N * (n_p * (6 * NQ[p] + 18 * (p + 1)) + 20 * (NQ[p] + 3 * (p + 1)))
    if c["kind"] == "rhs":
        return {"bytes": 2 * D + mesh, "flops": ops}
    if c["kind"] == "vjp":
        return {"bytes": 5 * D + 2 * mesh, "flops": 3 * ops}
    r = {"rk4": 1., "ssp3": 2. / 3, "ssp2": 0.5, "rk2": 0.5}[c["integrator"]]
    n = c["steps"] * STAGES[c["integrator"]]
    if c["kind"] == "adjoint":  # the stages, and per stage (state, weight) -> weight
        return {"bytes": n * ((5 + r) * D + 2 * mesh), "flops": n * 3 * ops}
    return {"bytes": n * ((2 + r) * D + mesh), "flops": n * ops}


# ------------------------------------------------------------ the scheme in plain torch

# points of the degree-2p rules on the triangle (Dunavant 1985) by their
# barycentric orbits: weight (of unit sum), then 1, 2 or 3 coordinates
RULES = (
    ((1.0,),),
    ((0.333333333333333, 0.166666666666666),),
    ((0.109951743655322, 0.091576213509771), (0.223381589678011, 0.445948490915965)),
    ((0.050844906370207, 0.063089014491502), (0.116786275726379, 0.249286745170910),
     (0.082851075618374, 0.636502499121399, 0.310352451033784)),
    ((0.144315607677787,), (0.095091634267285, 0.459292588292723),
     (0.103217370534718, 0.170569307751760), (0.032458497623198, 0.050547228317031),
     (0.027230314174435, 0.008394777409958, 0.728492392955404)),
    ((0.090817990382754,), (0.036725957756467, 0.485577633383657),
     (0.045321059435528, 0.109481575485037),
     (0.072757916845420, 0.141707219414880, 0.307939838764121),
     (0.028327242531057, 0.025003534762686, 0.246672560639903),
     (0.009421666963733, 0.009540815400299, 0.066803251012200)),
)
# where the rotating hill's speed is sampled for the time step
HILL_POINT = ((1 / 3, 1 / 3), (2 / 3, 1 / 6), (0.108103018168070, 0.445948490915965),
              (0.636502499121399, 0.310352451033784), (0.050547228317031, 0.898905543365938),
              (0.141707219414880, 0.550352941820999))


def _rule(p):
    pts, w = [], []
    for o in RULES[p]:
        if len(o) == 1:
            q = [(1 / 3, 1 / 3)]
        elif len(o) == 2:
            a, b = o[1], 1 - 2 * o[1]
            q = [(a, a), (a, b), (b, a)]
        else:
            a, b = o[1], o[2]
            d = 1 - a - b
            q = [(a, b), (b, a), (a, d), (d, a), (b, d), (d, b)]
        pts += q
        w += [o[0] / 2] * len(q)
    return np.array(pts), np.array(w)


@functools.lru_cache(maxsize=8)
def _basis(p):
    """orthonormal polynomials on the reference triangle: Gram-Schmidt of the
    graded monomials in exact arithmetic; rows of monomial coefficients"""
    mono = [(d - j, j) for d in range(p + 1) for j in range(d + 1)]
    f = math.factorial

    def inner(u, v):
        return sum(x * y * Fraction(f(a + k) * f(b + m), f(a + b + k + m + 2))
                   for x, (a, b) in zip(u, mono) if x for y, (k, m) in zip(v, mono) if y)
    rows, out = [], []
    for i in range(len(mono)):
        v = [Fraction(int(i == k)) for k in range(len(mono))]
        for u in rows:
            s = inner(v, u) / inner(u, u)
            v = [x - s * y for x, y in zip(v, u)]
        rows.append(v)
        n = inner(v, v)
        # the square root in extra digits
        root = Fraction(math.isqrt(n.numerator * n.denominator * 10**60), n.denominator * 10**30)
        out.append([x / root for x in v])
    return mono, out


def _poly(p, pts, d=None):
    """[n_p, points] basis values, or the derivative along r (0) or s (1)"""
    mono, co = _basis(p)
    out = np.zeros((len(mono), len(pts)))
    for j, (r, s) in enumerate(pts):
        r, s = Fraction(float(r)), Fraction(float(s))
        m = []
        for a, b in mono:
            if d is None:
                m.append(r**a * s**b)
            elif d == 0:
                m.append(a * r**(a - 1) * s**b if a else 0)
            else:
                m.append(b * r**a * s**(b - 1) if b else 0)
        for i in range(len(mono)):
            out[i, j] = float(sum(x * y for x, y in zip(co[i], m)))
    return out


@functools.lru_cache(maxsize=8)
def _tables(p):
    pts, w = _rule(p)
    x1, w1 = np.polynomial.legendre.leggauss(p + 1)
    sides = [[(0.5 + 0.5 * x, 0.) for x in x1], [((1 - x) / 2, (1 + x) / 2) for x in x1],
             [(0., 0.5 - 0.5 * x) for x in x1]]

    def t(a):
        return torch.tensor(np.asarray(a), dtype=F64, device=DEV)
    return dict(pts=pts, W=t(w), W1=t(w1), B=t(_poly(p, pts)), GX=t(_poly(p, pts, 0) * w),
                GY=t(_poly(p, pts, 1) * w), sides=sides, SIDE=t([_poly(p, q) for q in sides]))


def _sqrt32(a):
    return np.sqrt(np.asarray(a).astype(np.float32)).astype(np.float64)


class Plain:
    """The semi-discrete scheme of one case in torch float64."""

    def __init__(self, c, seed):
        self.c, self.T, self.N = c, _tables(c["p"]), L.NVARS[PHYS[c["physics"]]]
        self.phys, m = c["physics"], _mesh_of(c)
        self.K = m.K
        self.prob, self.prm = _problem(c, seed)

        def t(a, dt=F64):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=DEV)
        V = m.V
        self.V = t(V)
        self.xr, self.yr = t(V[2] - V[0]), t(V[3] - V[1])
        self.xs, self.ys = t(V[4] - V[0]), t(V[5] - V[1])
        self.J = t((V[2] - V[0]) * (V[5] - V[1]) - (V[4] - V[0]) * (V[3] - V[1]))
        a, b, d = (_sqrt32((V[i] - V[j])**2 + (V[i + 1] - V[j + 1])**2)
                   for i, j in ((0, 2), (2, 4), (0, 4)))
        k = 0.5 * (a + b + d)
        self.min_r = float((2 * _sqrt32(k * (k - a) * (k - b) * (k - d)) / k).min())
        # per element and local side: neighbour, its side, outward normal, length
        e, es = np.arange(m.K), m.elem_sides
        own = np.stack([np.where(m.left[es[q]] == e, m.lsn[es[q]], m.rsn[es[q]]) for q in range(3)])
        es = np.take_along_axis(es, np.argsort(own, axis=0), axis=0)
        role = m.left[es] != e
        dx, dy = m.side_xy[2] - m.side_xy[0], m.side_xy[3] - m.side_xy[1]
        ln = _sqrt32(dx * dx + dy * dy)
        # the left element walks its side from vertex lsn to the next one
        # (counter-clockwise), so its outward normal is (dy, -dx)
        i, j = m.lsn * 2, (m.lsn + 1) % 3 * 2
        turn = np.sign((V[j, m.left] - V[i, m.left]) * dx + (V[j + 1, m.left] - V[i + 1, m.left]) * dy)
        nx, ny = turn * dy / ln, -turn * dx / ln
        sg = np.where(role, -1., 1.)
        self.nx, self.ny, self.len = t(sg * nx[es]), t(sg * ny[es]), t(ln[es])
        nb = np.where(role, m.left[es], m.right[es])
        self.code = t(np.where(nb < 0, -nb, 0), torch.long)
        self.nb = t(np.where(nb < 0, e, nb), torch.long)
        self.nbls = t(np.where(role, m.lsn[es], np.maximum(m.rsn[es], 0)), torch.long)
        self.bnd = bool((nb < 0).any())
        eps = _eps(c, m.K, seed)
        self.eps = t(eps) if eps is not None else None
        self.gm, self.g = 1.4, 9.81

    def at(self, r, s):
        V = self.V
        return (V[2] * r + V[4] * s + V[0] * (1 - r - s), V[3] * r + V[5] * s + V[1] * (1 - r - s))

    # states of the problems
    def exact_state(self, x, y, t=0.0):
        pp, z = self.prm, torch.zeros_like(x)
        if self.prob == L.PROB_ADV_SINSIN:
            return torch.stack([torch.sin(2 * math.pi * (x - t)) * torch.sin(2 * math.pi * (y - t))])
        if self.prob == L.PROB_ADV_ROTHILL:
            co, si = math.cos(2 * math.pi * t), math.sin(2 * math.pi * t)
            X, Y = x * co + y * si, -x * si + y * co
            return torch.stack([5 * torch.exp(-((X - 0.2)**2 + Y * Y) / (2 * 0.15**2))])
        if self.prob == L.PROB_EULER_VORTEX:
            g = self.gm
            dx, dy = x - (pp[1] + pp[3] * t), y - (pp[2] + pp[4] * t)
            dx, dy = (q - 10 * torch.floor(q / 10 + 0.5) for q in (dx, dy))
            r2 = dx * dx + dy * dy
            f = pp[0] / (2 * math.pi) * torch.exp(0.5 * (1 - r2))
            u, v = pp[3] - f * dy, pp[4] + f * dx
            T = 1 - (g - 1) * pp[0]**2 / (8 * g * math.pi**2) * torch.exp(1 - r2)
            rho = T**(1 / (g - 1))
            return torch.stack([rho, rho * u, rho * v,
                                rho**g / (g - 1) + 0.5 * rho * (u * u + v * v)])
        if self.prob == L.PROB_EULER_SUPERSONIC:
            r, th = torch.sqrt(x * x + y * y), torch.atan(y / x)
            rho = (1 + 1.0125 * (1 - 1 / (r * r)))**2.5
            return torch.stack([rho, rho * torch.sin(th) * 2.25 / r, -rho * torch.cos(th) * 2.25 / r,
                                0.5 * rho * 2.25**2 / (r * r) + rho**1.4 / 1.4 / 0.4])
        if self.prob == L.PROB_SWE_BUMP:
            h = pp[0] + pp[1] * torch.exp(-((x - pp[2])**2 + (y - pp[3])**2) / (pp[5] * pp[4]**2))
            return torch.stack([h, z, z])
        return torch.stack([z, z, pp[0] * torch.exp(-((x - pp[1])**2 + (y - pp[2])**2) / pp[3]**2)])

    def project(self, f):
        c = 0.
        for j, (r, s) in enumerate(self.T["pts"]):
            u = f(*self.at(float(r), float(s)))
            c = c + self.T["W"][j] * self.T["B"][:, j][None, :, None] * u[:, None, :]
        return c.contiguous()

    # fluxes
    def velocity(self, r, s):
        """advection velocity at reference points [..., K]"""
        if self.prob != L.PROB_ADV_ROTHILL:
            return 1., 1.
        x, y = self.at(r, s)
        return -2 * math.pi * y, 2 * math.pi * x

    def flux(self, U, vel=None):
        if self.phys == "adv":
            return vel[0] * U, vel[1] * U
        z = torch.zeros_like(U[0])
        if self.phys in ("tm", "te"):
            return torch.stack([z, U[2], U[1]]), torch.stack([-U[2], z, -U[0]])
        u, v = U[1] / U[0], U[2] / U[0]
        if self.phys == "swe":
            q = 0.5 * self.g * U[0]**2
            return torch.stack([U[1], U[1] * u + q, U[1] * v]), torch.stack([U[2], U[2] * u, U[2] * v + q])
        p = (self.gm - 1) * (U[3] - 0.5 * (U[1] * u + U[2] * v))
        H = U[3] + p
        return (torch.stack([U[1], U[1] * u + p, U[1] * v, u * H]),
                torch.stack([U[2], U[2] * u, U[2] * v + p, v * H]))

    def speed(self, U, nx, ny):
        if self.phys == "tm":
            return torch.ones_like(U[0])
        vn = ((U[1] * nx + U[2] * ny) / U[0]).abs()
        if self.phys == "swe":
            return vn + torch.sqrt(self.g * U[0])
        p = (self.gm - 1) * (U[3] - 0.5 * (U[1]**2 + U[2]**2) / U[0])
        return vn + torch.sqrt(self.gm * p / U[0])

    def riemann(self, a, b, nx, ny, vel, ea, eb):
        if self.phys == "adv":
            an = vel[0] * nx + vel[1] * ny
            return torch.where(an > 0, a, b) * an
        if self.phys == "te":
            za, zb = torch.sqrt(1 / ea), torch.sqrt(1 / eb)
            ta, tb = -a[0] * ny + a[1] * nx, -b[0] * ny + b[1] * nx
            h = (za * a[2] + zb * b[2] + (ta - tb)) / (za + zb)
            e = (zb * ta + za * tb + za * zb * (a[2] - b[2])) / (za + zb)
            return torch.stack([-ny * h, nx * h, e])
        (fa, ga), (fb, gb) = self.flux(a), self.flux(b)
        F = 0.5 * ((fa + fb) * nx + (ga + gb) * ny)
        if self.c["flux"] == "roe":
            sa, sb = torch.sqrt(a[0]), torch.sqrt(b[0])
            u = (a[1] / sa + b[1] / sb) / (sa + sb)
            v = (a[2] / sa + b[2] / sb) / (sa + sb)
            cs = torch.sqrt(self.g * 0.5 * (a[0] + b[0]))
            un, ut = u * nx + v * ny, -u * ny + v * nx
            d = b - a
            dn, dt = d[1] * nx + d[2] * ny, -d[1] * ny + d[2] * nx
            w = (dn - un * d[0]) / cs
            k1 = (un - cs).abs() * 0.5 * (d[0] - w)
            k2 = un.abs() * (dt - ut * d[0])
            k3 = (un + cs).abs() * 0.5 * (d[0] + w)
            return F - 0.5 * torch.stack([k1 + k3, k1 * (u - cs * nx) - k2 * ny + k3 * (u + cs * nx),
                                          k1 * (v - cs * ny) + k2 * nx + k3 * (v + cs * ny)])
        lam = torch.maximum(self.speed(a, nx, ny), self.speed(b, nx, ny))
        return F + 0.5 * lam * (a - b)

    def ghost(self, a, k, j, t):
        """state outside boundary side k at its point j, [N, K] (meaningless at
        interior sides)"""
        r, s = self.T["sides"][k][j]
        nx, ny = self.nx[k], self.ny[k]
        if self.phys == "adv":
            return self.exact_state(*self.at(r, s), t)
        wx, wy = nx, ny
        if self.phys in ("tm", "te"):
            d = 2 * (a[0] * wx + a[1] * wy)
            return torch.stack([-a[0] + d * wx, -a[1] + d * wy, a[2]])
        if self.c["domain"] != "annulus":
            d = 2 * (a[1] * wx + a[2] * wy)
            return torch.cat([a[:1], (a[1] - d * wx)[None], (a[2] - d * wy)[None], a[3:]])
        x, y = self.at(r, s)
        q = torch.sqrt(x * x + y * y)
        q = torch.where(x * nx + y * ny < 0, -q, q)
        wx, wy = x / q, y / q
        m = a[1] * wy - a[2] * wx
        wall = torch.stack([a[0], m * wy, -m * wx, a[3]])
        return torch.where(self.code[k] == 1, wall, self.exact_state(x, y, t))

    def rhs(self, C, dt, t=0.0, eps=None):
        T, N, p = self.T, self.N, self.c["p"]
        if eps is None:
            eps = self.eps
        out = 0.
        for j, (r, s) in enumerate(T["pts"]):
            U = torch.einsum("nie,i->ne", C, T["B"][:, j])
            fx, fy = self.flux(U, self.velocity(float(r), float(s)) if self.phys == "adv" else None)
            ga, gb = fx * self.ys - fy * self.xs, fy * self.xr - fx * self.yr
            out = out + T["GX"][:, j][None, :, None] * ga[:, None] + T["GY"][:, j][None, :, None] * gb[:, None]
        tr = torch.stack([torch.einsum("nie,ij->nje", C, T["SIDE"][k]) for k in range(3)])
        tr = tr.permute(0, 3, 1, 2)  # [side, element, variable, point]
        for k in range(3):
            other = tr[self.nbls[k], self.nb[k]]
            nx, ny = self.nx[k], self.ny[k]
            ea, eb = (eps, eps[self.nb[k]]) if eps is not None else (None, None)
            for j in range(p + 1):
                a, b = tr[k, :, :, j].t(), other[:, :, p - j].t()
                if self.bnd:
                    b = torch.where(self.code[k] > 0, self.ghost(a, k, j, t), b)
                vel = self.velocity(*T["sides"][k][j]) if self.phys == "adv" else None
                F = self.riemann(a, b, nx, ny, vel, ea, eb) * (0.5 * T["W1"][j] * self.len[k])
                out = out - T["SIDE"][k][:, j][None, :, None] * F[:, None]
        out = out * (dt / self.J)
        if eps is not None:
            out = torch.cat([out[:2] / eps, out[2:]])
        return out

    def dt(self, C, cfl):
        U = C[:, 0] * math.sqrt(2.0)
        if self.phys == "adv":
            v = self.velocity(*HILL_POINT[self.c["p"]])
            lam = float(torch.sqrt(torch.as_tensor(v[0]**2 + v[1]**2, dtype=F64)).max())
        elif self.phys in ("tm", "te"):
            lam = 1. if self.eps is None else float((1 / torch.sqrt(self.eps)).max())
        else:
            s = torch.sqrt(U[1]**2 + U[2]**2) / U[0]
            if self.phys == "swe":
                lam = float((s + torch.sqrt(self.g * U[0])).max())
            else:
                p = (self.gm - 1) * (U[3] - 0.5 * (U[1]**2 + U[2]**2) / U[0])
                lam = float((s + torch.sqrt(self.gm * p / U[0])).max())
        return cfl * self.min_r / lam / (2 * self.c["p"] + 1)

    def limit(self, C):
        """the p = 1 slope limiter (on every mean and side value)"""
        m = C[:, 0] * math.sqrt(2.0)
        lo = hi = m
        for k in range(3):
            v = m[:, self.nb[k]]
            lo, hi = torch.minimum(lo, v), torch.maximum(hi, v)
        al = torch.ones_like(m)
        for k in range(3):
            for j in range(2):
                d = torch.einsum("nie,i->ne", C, self.T["SIDE"][k][:, j]) - m
                q = torch.where(d > 0, (m - lo) / d, torch.where(d < 0, (m - hi) / d, 1.))
                al = torch.minimum(al, q)
        al = al.clamp(min=0.)
        return torch.stack([C[:, 0], C[:, 1] * al, C[:, 2] * al], dim=1)

    def step(self, C, dt, t, eps=None):
        """one step (stage times count from the step's end, as the solver's)"""
        lim = self.limit if self.c["limiter"] else (lambda x: x)

        def f(u, cs):
            return lim(self.rhs(u, dt, t + dt + cs * dt, eps))
        k = f(C, 0.)
        if self.c["integrator"] == "rk4":
            k2 = f(C + 0.5 * k, 0.5)
            k3 = f(C + 0.5 * k2, 0.5)
            k4 = f(C + k3, 1.)
            return lim(C + (k / 6 + k2 / 3 + k3 / 3 + k4 / 6))
        if self.c["integrator"] == "rk2":
            return lim(C + f(C + 0.5 * k, 0.5))
        u = C + k
        if self.c["integrator"] == "ssp2":
            return lim(0.5 * C + 0.5 * u + 0.5 * f(u, 1.))
        u = 0.75 * C + 0.25 * u + 0.25 * f(u, 1.)
        return lim(C / 3 + 2 / 3 * u + 2 / 3 * f(u, 0.5))

    def objective(self, C):
        J, W = self.J, self.T["W"]
        U = torch.einsum("nie,ij->nje", C, self.T["B"])
        if self.phys == "te":
            cx, cy = (self.V[0] + self.V[2] + self.V[4]) / 3, (self.V[1] + self.V[3] + self.V[5]) / 3
            x0, x1, y0, y1, n = PATCH
            inside = (cx >= x0) & (cx <= x1) & (cy >= y0) & (cy <= y1)
            return (torch.where(inside, J, 0.) * torch.einsum("je,j->e", U[n]**2, W)).sum()
        p = (self.gm - 1) * (U[3] - 0.5 * (U[1]**2 + U[2]**2) / U[0])
        return (J * torch.einsum("je,j->e", -U[0] * (torch.log(p) - self.gm * torch.log(U[0])), W)).sum()


def _initial(c, seed):
    """the projected initial state with a seeded smooth perturbation"""
    P = Plain(c, seed)
    r = np.random.default_rng(seed + 1)
    a, ph = r.uniform(0.005, 0.02), r.uniform(0, 2 * math.pi, 2)
    w = 2 * math.pi * (0.1 if c["physics"] == "euler" and c["domain"] == "periodic" else 1.)

    def f(x, y):
        return P.exact_state(x, y) * (1 + a * torch.sin(w * (2 * x + y) + ph[0])
                                      * torch.sin(w * (y - 2 * x) + ph[1]))
    return P.project(f)


def _adjoint_dt(c, seed, u):
    return Plain(c, seed).dt(u, c["cfl"] or (0.7 if c["integrator"] == "rk2" else 0.5))


def exact(case, seed):
    c = case
    if c["kind"] == "ensemble":
        out = []
        for ci, si in _instances(c, seed):
            # an instance's perturbation and bump are its own, as prepare() sets them
            out.append(_run_exact(ci, si)["c"])
        return out
    P = Plain(c, seed)
    u = _initial(c, seed)
    if c["kind"] == "rhs":
        return P.rhs(u, 0.01)
    if c["kind"] == "vjp":
        u.requires_grad_(True)
        k = P.rhs(u, 0.01)
        (gu,) = torch.autograd.grad(k, u, _weights(c, seed, u.shape))
        return {"k": k.detach(), "gu": gu}
    if c["kind"] == "steps":
        return _run_exact(c, seed)
    dt = _adjoint_dt(c, seed, u)
    leaves = [u.requires_grad_(True)] + ([P.eps.requires_grad_(True)] if P.eps is not None else [])
    C, t = u, 0.
    for _ in range(c["steps"]):
        C = torch.utils.checkpoint.checkpoint(P.step, C, dt, t, P.eps, use_reentrant=False)
        t += dt
    J = P.objective(C)
    return {"J": J.detach(), "g": list(torch.autograd.grad(J, leaves))}


def _run_exact(c, seed):
    P = Plain(c, seed)
    C, t = _initial(c, seed), 0.
    cfl = c["cfl"] or (0.7 if c["integrator"] == "rk2" else 0.5)
    if c["limiter"]:
        C = P.limit(C)
    with torch.no_grad():
        for _ in range(c["steps"]):
            dt = P.dt(C, cfl)
            C = P.step(C, dt, t)
            t += dt
    return {"c": C, "t": t}
