"""The kernels of larger meshes (a thread or four lanes per element), on meshes
just above the sizes up to which the point-parallel ones run: stored traces,
the vector-Jacobian products, the Runge-Kutta terms that they add for a whole
gradient, and resident segments; and the point-parallel kernels' narrow form at
p = 2, near the top of its range.  The sizes are read from the rules' tables in
the sources, so a table that moves takes these meshes with it."""
import os
import re

import numpy as np
import pytest
import torch

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from dgcuda_amd.solver import Solver
from tests.helpers import CASES, make_pair, rel_l2
from tests.tape import TABLEAUS, Tape

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = 1e-12
PH_ROWS = {L.ADVECTION: 0, L.EULER: 1, L.SWE: 2, L.MAXWELL_TM: 3, L.MAXWELL_TE: 3}


def _table(source, function):
    txt = open(os.path.join(ROOT, "dgcuda_amd", "csrc", source)).read()
    body = txt[txt.index("int %s(" % function):]
    body = body[body.index("{{"):body.index("}};") + 2]
    return [[int(x) for x in re.findall(r"\d+", row)] for row in re.findall(r"\{([\d, \n]+)\}", body)]


def top_stage(physics, p):
    n = L.NVARS[physics]
    return _table("dg_kernels.hip", "small_max_k")[0 if n == 1 else n - 2][p]


def top_vjp(physics, p, eps=False):
    return _table("dg_adjoint.hip", "small_max_vjp")[4 if eps else PH_ROWS[physics]][p]


def above(*tops):
    """squares per side of the smallest box above these many triangles"""
    n = int(np.sqrt(max(tops) / 2))
    while 2 * n * n <= max(tops):
        n += 1
    return n


def _mesh(n, periodic=False, **kw):
    return M.structured(n, periodic=periodic, jitter=0.2, seed=7, **kw)


def _pair(physics, p, n, periodic=False, bc=(-1, -1, -1, -1), **kw):
    mesh = _mesh(n, periodic, bc=bc)
    eps = np.random.default_rng(3).uniform(1.0, 4.0, mesh.K)
    s, o = make_pair(physics, p, mesh, eps_elem=eps if physics == L.MAXWELL_TE else None, **kw)
    s.project_ic()
    o.project_ic()
    return s, o


# ------------------------------------------------------------ stored traces


def _traces(p, integrator, gather, mesh):
    prob, prm, fl = CASES[L.EULER]
    if gather:
        os.environ["DG_STAGE_GATHER"] = "1"
    try:
        s = Solver(L.EULER, p, integrator=integrator, flux=fl, cfl=0.5, problem=prob,
                   problem_params=prm)
    finally:
        os.environ.pop("DG_STAGE_GATHER", None)
    return s.set_mesh(mesh).project_ic()


def _held(s):
    """device memory that goes with the handle"""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    s.close()
    return torch.cuda.mem_get_info()[0] - before


@pytest.mark.parametrize("p,integrator,periodic,flagged", [
    (4, L.SSPRK3, True, False), (4, L.RK4, False, False), (4, L.SSPRK2, True, False),
    (5, L.SSPRK3, False, False), (4, L.SSPRK3, True, True), (5, L.RK2MID, False, True)])
def test_stored_traces_equal_the_gather_path(p, integrator, periodic, flagged):
    """as tests/test_gpu_traces.py, to rounding, on a mesh that stores traces
    (the handle holds them: three arrays of 12 (p + 1) doubles an element)"""
    mesh = _mesh(above(top_stage(L.EULER, p)), periodic)
    out, held = [], []
    for gather in (True, False):
        s = _traces(p, integrator, gather, mesh)
        u = s.coeffs()
        if flagged:
            u[:, 1:, ::5] *= 400.0  # these contribute their means only
            s.set_coeffs(u)
        kw = dict(dt=1e-4) if flagged else {}
        t1, _ = s.step(7, **kw)         # graphs of 4, 2 and 1 steps
        t2, dt = s.step(5, t=t1, **kw)  # a second run starts from a fresh fill
        out.append((t2, dt, s.coeffs()))
        held.append(_held(s))
    tr = 3 * 12 * (p + 1) * 8 * mesh.K
    (tb, db, cb), (ta, da, ca) = out
    print("p", p, "K", mesh.K, "rel", rel_l2(ca, cb), "dt", da, db, "held", held, "traces", tr,
          flush=True)
    assert held[1] - held[0] > 0.7 * tr
    assert np.isfinite(ca).all() and np.isfinite(cb).all()
    assert abs(ta - tb) <= 1e-14 * abs(tb) and abs(da - db) <= 1e-13 * abs(db)
    assert rel_l2(ca, cb) < 1e-13


@pytest.mark.parametrize("p,integrator", [(4, L.SSPRK3), (4, L.RK4), (5, L.SSPRK2)])
def test_stored_traces_parity_with_the_oracle(p, integrator):
    s, o = _pair(L.EULER, p, above(top_stage(L.EULER, p)), periodic=True, integrator=integrator,
                 cfl=0.2)
    u = o.coeffs()
    u[:, 1:, ::41] *= 400.0
    s.set_coeffs(u)
    o.set_coeffs(u)
    ts, _ = s.step(3, dt=1e-4)
    rc, to, _ = o.run(3, dt=1e-4)
    r = rel_l2(s.coeffs(), o.coeffs())
    print("traces p", p, "K", s.K, "rel", r, flush=True)
    assert rc == 0 and abs(ts - to) <= 1e-13 * abs(to) and r < TOL
    s.close()


# ------------------------------------------------------------ VJPs and gradients


def _directions(u, r):
    """unit directions: everywhere, the first and last blocks, every 97th"""
    K = u.shape[2]
    masks = [np.ones(K, bool), np.zeros(K, bool), np.zeros(K, bool)]
    masks[1][:5] = masks[1][-70:] = True
    masks[2][::97] = True
    for m in masks:
        v = r.standard_normal(u.shape) * m
        yield v / np.linalg.norm(v), m


ROE = dict(flux=L.FLUX_ROE)
INFLOW = dict(problem=L.PROB_EULER_VORTEX, params=(5.0, 0.5, 0.5, 1.0, 1.0, 1.0),
              bc=(-3, -2, -3, -2))
HILL = dict(problem=L.PROB_ADV_ROTHILL, params=(), bc=(-3, -3, -2, -3))


@pytest.mark.parametrize("physics,p,kw", [
    (L.ADVECTION, 1, {}), (L.ADVECTION, 2, HILL), (L.ADVECTION, 5, {}), (L.EULER, 2, INFLOW),
    (L.EULER, 3, {}), (L.EULER, 4, {}), (L.EULER, 5, INFLOW), (L.SWE, 1, ROE), (L.SWE, 3, ROE),
    (L.SWE, 5, {}), (L.MAXWELL_TM, 2, {}), (L.MAXWELL_TE, 1, {}), (L.MAXWELL_TE, 3, {}),
    (L.MAXWELL_TE, 5, {})])
def test_wide_vjp(physics, p, kw):
    """<g, J v> = <J^T g, v>, v everywhere or on few elements, g on those and
    their neighbours: J v is the oracle's central difference along a unit v
    (step 1e-4: truncation ~1e-8 of a smooth second derivative, rounding
    ~1e-12)"""
    s, o = _pair(physics, p, above(top_vjp(physics, p)), **kw)
    r = np.random.default_rng(p)
    u = o.coeffs()
    u = u + 0.01 * r.standard_normal(u.shape) / np.sqrt(u.shape[1])
    if physics == L.SWE:
        u[0, 0] += 1.0
    print("physics", physics, "p", p, "K", s.K, flush=True)
    h = 1e-4
    for v, m in _directions(u, r):
        jv = (o.eval_rhs(u + h * v, dt=0.01) - o.eval_rhs(u - h * v, dt=0.01)) / (2 * h)
        g = r.standard_normal(u.shape) * (np.abs(jv).max(axis=(0, 1)) > 0)
        gu = s.adjoint_rhs(u, g, dt=0.01)
        fd, scale = np.vdot(g, jv), np.linalg.norm(gu[:, :, m])
        print("  on", int(m.sum()), "fd", fd, "vjp", np.vdot(gu, v), "scale", scale)
        assert abs(np.vdot(gu, v) - fd) < 1e-6 * scale
    s.close()


@pytest.mark.parametrize("physics,p,integrator,periodic", [
    (L.EULER, 4, L.SSPRK3, True), (L.EULER, 4, L.RK4, False), (L.EULER, 5, L.SSPRK2, True),
    (L.EULER, 2, L.SSPRK3, True), (L.EULER, 3, L.RK2MID, False), (L.MAXWELL_TE, 3, L.RK4, False),
    (L.MAXWELL_TE, 5, L.SSPRK3, False)])
def test_wide_gradient_matches_the_tape(physics, p, integrator, periodic):
    """as tests/test_gpu_adjoint.py, the whole gradient to rounding, with one
    recomputed segment and one that the forward pass records"""
    te = physics == L.MAXWELL_TE
    mesh = _mesh(above(top_vjp(physics, p, te), top_stage(physics, p)), periodic)
    rng = np.random.default_rng(20 + p)
    eps = rng.uniform(1, 4, mesh.K) if te else None
    if te:
        s, o = make_pair(physics, p, mesh, integrator=integrator, eps_elem=eps)
        kind, prm = L.OBJ_PATCH_SQ, (0.5, 0.9, 0.4, 0.8, 2)
    else:
        prm_v = (5.0, 0.5, 0.5, 1.0, 1.0, 1.0) if periodic else (5.0, 0.5, 0.5, 0.0, 0.0, 1.0)
        s, o = make_pair(physics, p, mesh, integrator=integrator, params=prm_v)
        kind, prm = L.OBJ_ENTROPY, ()
    o.project_ic()
    u0 = o.coeffs() * (1.0 + 0.02 * rng.standard_normal((o.N, o.n_p, o.K)))
    if te:
        u0[:2] = 0.05 * np.abs(u0[2]).max() * rng.standard_normal(u0[:2].shape)
    dt = 0.1 * s.info().min_r / (2 * p + 1)
    s.set_objective(kind, prm)
    s.set_coeffs(u0)
    print("tape", physics, p, "K", mesh.K, "integrator", integrator, flush=True)
    J, gu, ge = s.adjoint_solve(3, dt, every=2, want_eps=te)
    Jt, gut, get = Tape(o, mesh, physics).gradient(u0, 3, dt, integrator, kind, prm, eps)
    print("  J", J, Jt, "grad u0 rel", rel_l2(gu, gut), "worst", np.abs(gu - gut).max() /
          np.abs(gut).max(), "grad eps rel", rel_l2(ge, get) if te else None)
    assert abs(J - Jt) <= 1e-12 * abs(Jt)
    assert rel_l2(gu, gut) <= 1e-10 and np.abs(gu - gut).max() <= 1e-10 * np.abs(gut).max()
    if te:
        assert rel_l2(ge, get) <= 1e-10
    s.close()


C_NODES = {L.RK4: (0, 0.5, 0.5, 1.0), L.RK2MID: (0, 0.5), L.SSPRK2: (0, 1.0), L.SSPRK3: (0, 1.0, 0.5)}


@pytest.mark.parametrize("physics,p,integrator,kw", [
    (L.SWE, 2, L.SSPRK3, ROE), (L.SWE, 4, L.RK4, ROE), (L.EULER, 2, L.RK4, INFLOW),
    (L.EULER, 4, L.SSPRK3, INFLOW), (L.ADVECTION, 1, L.RK2MID, HILL),
    (L.ADVECTION, 2, L.SSPRK3, HILL), (L.ADVECTION, 5, L.RK4, {}), (L.MAXWELL_TM, 1, L.SSPRK3, {}),
    (L.MAXWELL_TE, 1, L.SSPRK2, {})])
def test_wide_gradient_is_the_transposed_tableau(physics, p, integrator, kw):
    """the gradient of a linear objective is the integrator's tableau
    transposed over single vector-Jacobian products at its stage states (both
    are public calls of their own): to rounding, in every entry"""
    s, _ = _pair(physics, p, above(top_vjp(physics, p), top_stage(physics, p)),
                 integrator=integrator, **kw)
    a, b = TABLEAUS[integrator]
    c, S, n = C_NODES[integrator], len(b), 3
    dt = 0.1 * s.info().min_r / (2 * p + 1)
    r = np.random.default_rng(p)
    u0 = s.coeffs()
    u0 = u0 + 0.01 * r.standard_normal(u0.shape) / np.sqrt(u0.shape[1])
    w = r.standard_normal(u0.shape)
    s.set_objective(L.OBJ_LINEAR, weights=w)
    s.set_coeffs(u0)
    print("tableau", physics, p, "K", s.K, "integrator", integrator, flush=True)
    J, gu, _ = s.adjoint_solve(n, dt, every=2)
    u, stages = u0, []
    for q in range(n):
        ks, us = [], []
        for i in range(S):
            us.append(u + sum((a[i][j] * ks[j] for j in range(i) if a[i][j]), 0.0))
            ks.append(s.eval_rhs(us[i], t=(q + 1 + c[i]) * dt, dt=dt))
        u = u + sum(b[i] * ks[i] for i in range(S) if b[i])
        stages.append(us)
    g = w
    for q in reversed(range(n)):
        ls = [None] * S
        for i in reversed(range(S)):
            gk = b[i] * g + sum((a[j][i] * ls[j] for j in range(i + 1, S) if a[j][i]), 0.0)
            ls[i] = s.adjoint_rhs(stages[q][i], gk, t=(q + 1 + c[i]) * dt, dt=dt)
        g = g + sum(ls)
    Jt = np.vdot(w, u)
    print("  J", J, Jt, "rel", rel_l2(gu, g), "worst", np.abs(gu - g).max())
    assert abs(J - Jt) <= 1e-13 * np.abs(w * u).sum()
    # (an entry sums some 100 terms of at most max|g|)
    assert rel_l2(gu, g) < TOL and np.abs(gu - g).max() <= 100 * TOL * np.abs(g).max()
    s.close()


@pytest.mark.parametrize("physics,p,integrator", [(L.EULER, 4, L.SSPRK3), (L.SWE, 2, L.RK4)])
def test_wide_resident_segments_match_the_recompute(physics, p, integrator):
    from tests.test_gpu_adjoint import _one_resident_gb, _solve_with_store
    s, _ = _pair(physics, p, above(top_vjp(physics, p), top_stage(physics, p)), periodic=True,
                 integrator=integrator, cfl=0.2)
    u0 = s.coeffs()
    s.set_objective(L.OBJ_LINEAR, weights=np.random.default_rng(1).standard_normal(u0.shape))
    dt = 0.1 * s.info().min_r / (2 * p + 1)
    one = _one_resident_gb(s.K, s.N, s.n_p, len(TABLEAUS[integrator][1]), 7, 3, False)
    print("resident", physics, p, "K", s.K, flush=True)
    out = [_solve_with_store(s, u0, 7, dt, 3, None, gb) for gb in (None, one, 1000.0)]
    assert [x[3] for x in out] == [0, 1, 3]
    for x in out[1:]:
        assert x[0] == out[0][0] and np.array_equal(x[1], out[0][1])
    s.close()


# ------------------------------------------------------------ p = 2, narrow


@pytest.mark.parametrize("physics", [L.ADVECTION, L.EULER, L.SWE, L.MAXWELL_TM, L.MAXWELL_TE])
def test_narrow_blocks_at_p2(physics):
    """p = 2 from 513 blocks of 16 elements on: 256 threads a block instead of
    384, in the stage and in the VJP, with a ragged last block"""
    top = min(top_stage(physics, 2), top_vjp(physics, 2))
    for nx, ny in ((64, 65), (above(top) - 1, (top // 2) // (above(top) - 1))):
        mesh = M.structured(nx, ny, periodic=False, jitter=0.2, seed=5)
        assert 512 * 16 < mesh.K <= top
        eps = np.random.default_rng(3).uniform(1.0, 4.0, mesh.K)
        s, o = make_pair(physics, 2, mesh, integrator=L.RK4, cfl=0.3,
                         eps_elem=eps if physics == L.MAXWELL_TE else None)
        o.project_ic()
        r = np.random.default_rng(nx)
        u = o.coeffs() * (1.0 + 0.05 * r.standard_normal(o.shape))
        print("narrow", physics, "K", mesh.K, flush=True)
        h = 1e-4
        for v, m in _directions(u, r):
            jv = (o.eval_rhs(u + h * v, dt=0.01) - o.eval_rhs(u - h * v, dt=0.01)) / (2 * h)
            g = r.standard_normal(u.shape) * (np.abs(jv).max(axis=(0, 1)) > 0)
            gu = s.adjoint_rhs(u, g, dt=0.01)
            assert abs(np.vdot(gu, v) - np.vdot(g, jv)) < 1e-6 * np.linalg.norm(gu[:, :, m])
        if physics in (L.EULER, L.SWE):
            u[:, 1:, ::41] *= 400.0  # elements that contribute their means only
        assert rel_l2(s.eval_rhs(u, t=0.1, dt=0.01), o.eval_rhs(u, t=0.1, dt=0.01)) < TOL
        s.set_coeffs(u)
        o.set_coeffs(u)
        t, _ = s.step(3, dt=1e-4)
        rc, to, _ = o.run(3, dt=1e-4)
        x = rel_l2(s.coeffs(), o.coeffs())
        print("  steps rel", x)
        assert rc == 0 and abs(t - to) <= 1e-13 * to and x < TOL
        s.close()
