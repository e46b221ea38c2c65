"""Moving boundary data on meshes that run the point-parallel stage, for the
systems whose stage does not evaluate them itself: any system may take the
vortex's or the travelling wave's states on its inflow and outflow sides.  Runs
against the oracle at the parity tests' bar, 1e-12 relative L2 (with the data of
the run's start in place of a stage's, one step is off by 2.5e-7 to 6e-4)."""
import numpy as np
import pytest

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair, rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-12
VORTEX = (5.0, 0.5, 0.5, 1.0, 1.0, 0.0)


def _pair(physics, p, nx, ny, problem, **kw):
    mesh = M.structured(nx, ny, periodic=False, jitter=0.2, seed=3, bc=(-3, -3, -2, -1))
    eps = np.random.default_rng(3).uniform(1.0, 4.0, mesh.K)
    s, o = make_pair(physics, p, mesh, problem=problem,
                     params=VORTEX if problem == L.PROB_EULER_VORTEX else (), cfl=0.3,
                     eps_elem=eps if physics == L.MAXWELL_TE else None, **kw)
    s.project_ic()
    o.project_ic()
    return s, o


# (5, 46, 47): more blocks than a step's first stage closes by itself
@pytest.mark.parametrize("physics,p,nx,ny,problem,integrator,limiter", [
    (L.SWE, 1, 7, 9, L.PROB_EULER_VORTEX, L.RK4, True),
    (L.SWE, 0, 3, 5, L.PROB_EULER_VORTEX, L.SSPRK2, False),
    (L.SWE, 2, 7, 9, L.PROB_EULER_VORTEX, L.RK4, False),
    (L.SWE, 5, 46, 47, L.PROB_EULER_VORTEX, L.SSPRK3, False),
    (L.MAXWELL_TM, 3, 7, 9, L.PROB_ADV_SINSIN, L.SSPRK3, False),
    (L.MAXWELL_TE, 4, 7, 9, L.PROB_EULER_VORTEX, L.RK2MID, False),
    (L.EULER, 2, 7, 9, L.PROB_EULER_VORTEX, L.SSPRK3, False),
    (L.EULER, 1, 7, 9, L.PROB_EULER_VORTEX, L.RK4, True)])
def test_runs_with_moving_boundary_data(physics, p, nx, ny, problem, integrator, limiter):
    s, o = _pair(physics, p, nx, ny, problem, integrator=integrator, limiter=limiter)
    print("moving", physics, p, s.K, problem, integrator, limiter, flush=True)
    t = to = 0.0
    for n in (1, 6):  # launched directly, then as graphs of 4 and 2 steps
        t, dt = s.step(n, t=t)
        rc, to, _, _, dto = o.run_until(max_steps=n, t0=to)
        r = rel_l2(s.coeffs(), o.coeffs())
        print("  steps", n, "rel", r, "t", t, to)
        assert rc == 0 and abs(t - to) <= 1e-13 * to and abs(dt - dto) <= 1e-13 * dto
        assert r < TOL
    t, n, _ = s.run(t=t, t_end=t + 2.5 * dt)  # the third step is shortened
    rc, to, no, _, _ = o.run_until(t0=to, t_end=to + 2.5 * dto)
    assert rc == 0 and n == no == 3 and abs(t - to) <= 1e-13 * to
    assert rel_l2(s.coeffs(), o.coeffs()) < TOL
    # the caller's states do not move, and the problem's do again
    _, _, x, _ = s.boundary_points()
    s.set_boundary_states(s.boundary_states(0.25))
    s.step(2, t=t)
    s.set_boundary_states(None)
    c = s.coeffs()
    o.set_coeffs(c)
    t, _ = s.step(3, t=t)
    rc, to, _, _, _ = o.run_until(max_steps=3, t0=to)
    assert rc == 0 and abs(t - to) <= 1e-13 * to and rel_l2(s.coeffs(), o.coeffs()) < TOL
    s.close()


@pytest.mark.parametrize("physics,p", [(L.SWE, 2), (L.MAXWELL_TE, 3)])
def test_gradient_with_moving_boundary_data(physics, p):
    """the adjoint's forward map is the run of steps, whatever its segments:
    the objective is that of the stepped state, the gradient the same for every
    checkpoint distance and that of central differences (step 1e-5 of a state
    of order one: truncation 1e-10, rounding 1e-11)"""
    s, _ = _pair(physics, p, 5, 6, L.PROB_EULER_VORTEX, integrator=L.RK4)
    u0, dt, n = s.coeffs(), 2e-3, 6
    r = np.random.default_rng(5)
    s.set_objective(L.OBJ_LINEAR, weights=r.standard_normal(u0.shape))

    def J(u):
        s.set_coeffs(u)
        s.step(n, dt=dt)
        return s.objective()
    j0 = J(u0)
    grads = []
    for every in (1, 4, 6):
        s.set_coeffs(u0)
        j, g, _ = s.adjoint_solve(n, dt, every=every)
        print("gradient", physics, p, "every", every, j, j0, flush=True)
        assert abs(j - j0) <= 1e-12 * np.linalg.norm(u0) * np.sqrt(u0.size)
        grads.append(g)
    assert rel_l2(grads[0], grads[1]) < TOL and rel_l2(grads[2], grads[1]) < TOL
    v = r.standard_normal(u0.shape)
    fd = (J(u0 + 1e-5 * v) - J(u0 - 1e-5 * v)) / 2e-5
    assert abs(np.vdot(grads[0], v) - fd) < 1e-6 * np.linalg.norm(grads[0]) * np.linalg.norm(v)
    s.close()
