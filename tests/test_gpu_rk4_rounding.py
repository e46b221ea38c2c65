"""A classical Runge-Kutta step adds its increment to the state with one
rounding: k1 .. k4 are summed at the increment's own scale, whatever the size
of the state beside it.  With a step of dt = 1e-10 the increment is far below
the state, so the step is u + (k1 + 2 k2 + 2 k3 + k4) / 6 (here from the
library's right-hand sides, summed in 80 bits) to half a unit in the last
place, plus the rounding of the k themselves: the residual's terms are below
T = 100 dt max|u| / min_r in sum, so 64 eps T (below 1e-3 of a unit of the
state) covers it.  From the rounded stage states it is up to a whole unit off."""
import numpy as np
import pytest

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair

pytestmark = pytest.mark.gpu


# either side of the meshes that run the point-parallel stage
@pytest.mark.parametrize("physics,p,K", [
    (L.ADVECTION, 1, 338), (L.ADVECTION, 1, 12800), (L.ADVECTION, 3, 338), (L.ADVECTION, 4, 13122),
    (L.MAXWELL_TM, 2, 338), (L.MAXWELL_TM, 2, 13122), (L.MAXWELL_TE, 3, 338),
    (L.MAXWELL_TE, 3, 17298), (L.EULER, 2, 338), (L.SWE, 3, 17298)])
def test_one_rounding_per_step(physics, p, K):
    n = int(np.sqrt(K // 2))
    mesh = M.structured(n, periodic=True, jitter=0.2, seed=7)
    assert mesh.K == K
    eps = np.random.default_rng(3).uniform(1.0, 4.0, K) if physics == L.MAXWELL_TE else None
    s, _ = make_pair(physics, p, mesh, integrator=L.RK4, eps_elem=eps)
    s.project_ic()
    u = s.coeffs()
    r = np.random.default_rng(p)
    if physics in (L.EULER, L.SWE):
        u = u * (1.0 + 1e-3 * r.standard_normal(u.shape))
    else:
        u[:, 0] += r.uniform(0.5, 1.0, u[:, 0].shape)
    dt = 1e-10
    k1 = s.eval_rhs(u, dt=dt)
    k2 = s.eval_rhs(u + 0.5 * k1, dt=dt)
    k3 = s.eval_rhs(u + 0.5 * k2, dt=dt)
    k4 = s.eval_rhs(u + k3, dt=dt)
    x = np.longdouble
    exact = x(u) + (x(k1) + 2 * x(k2) + 2 * x(k3) + x(k4)) / 6
    s.set_coeffs(u)
    s.step(1, dt=dt)
    out = s.coeffs()
    err = np.abs(x(out) - exact)
    T = 100.0 * dt * np.abs(u).max() / s.info().min_r
    bound = 0.5 * np.spacing(np.abs(out)) + 64 * 2.0 ** -52 * T
    print("physics", physics, "p", p, "K", K, "largest error / bound", float((err / bound).max()),
          "in units of the last place", float((err / np.spacing(np.abs(out)))[:, 0].max()),
          "beyond", int((err > bound).sum()), "of", err.size, flush=True)
    assert (err <= bound).all()
    s.close()
