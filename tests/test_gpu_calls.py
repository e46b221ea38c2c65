"""Calls on device arrays: read and written in place where they can be, through
the handle's buffers where they overlap or are host data, with the same result
to the bit (the same kernels on the same values); and state that a handle keeps
between calls: boundary data, captured steps, the adjoint's buffers."""
import ctypes

import numpy as np
import pytest

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics,p,n", [(L.EULER, 1, 5), (L.SWE, 2, 8), (L.EULER, 4, 60),
                                         (L.MAXWELL_TE, 0, 4), (L.ADVECTION, 3, 7)])
def test_device_arrays_in_place_and_overlapping(physics, p, n):
    import torch
    mesh = M.structured(n, periodic=False, jitter=0.2, seed=4)
    s, o = make_pair(physics, p, mesh)
    s.project_ic()
    u = s.coeffs() * (1.0 + 0.02 * np.random.default_rng(n).standard_normal(s.shape))
    g = np.random.default_rng(n + 1).standard_normal(s.shape)
    print("calls", physics, p, s.K, flush=True)
    k, gu = s.eval_rhs(u, t=0.1, dt=0.01), s.adjoint_rhs(u, g, t=0.1, dt=0.01)
    # an odd offset (8-byte aligned only), then the output over the input's tail
    buf = torch.zeros(2 * s.size + 1, dtype=torch.float64, device="cuda")
    ud, gd = buf[1:s.size + 1], torch.from_numpy(g).cuda()
    ud.copy_(torch.from_numpy(u).reshape(-1))
    out = torch.empty(s.shape, dtype=torch.float64, device="cuda")
    s.eval_rhs(ud, t=0.1, dt=0.01, out=out)
    assert np.array_equal(out.cpu().numpy(), k)
    assert np.array_equal(s.adjoint_rhs(ud, gd, t=0.1, dt=0.01).cpu().numpy(), gu)
    addr = [ctypes.c_void_p(x) for x in (ud.data_ptr(), gd.data_ptr(),
                                         ud.data_ptr() + 8 * (s.size // 2))]
    for call, want in ((lambda: s.lib.dg_adjoint_rhs(s.h, addr[0], 0.1, 0.01, addr[1], addr[2],
                                                     L.DEVICE), gu),
                       (lambda: s.lib.dg_eval_rhs(s.h, addr[0], 0.1, 0.01, addr[2], L.DEVICE), k)):
        ud.copy_(torch.from_numpy(u).reshape(-1))
        torch.cuda.synchronize()
        s._chk(call())
        a = 1 + s.size // 2
        assert np.array_equal(buf[a:a + s.size].cpu().numpy(), want.reshape(-1))
    s.close()


def test_boundary_states_between_runs():
    """captured steps with a moving inflow, then the caller's states, then the
    problem's again: each run equals a fresh solver's from the same state"""
    mesh = M.structured(6, lx=2.0, ly=2.0, x0=-1.0, y0=-1.0, periodic=False, jitter=0.2, seed=3,
                        bc=(-3, -3, -2, -3))

    def fresh():
        return make_pair(L.ADVECTION, 2, mesh, problem=L.PROB_ADV_ROTHILL, params=())[0]
    s = fresh().project_ic()
    _, _, x, _ = s.boundary_points()
    U = np.random.default_rng(1).uniform(0.0, 1.0, x.shape + (1,))
    t, _ = s.step(3)
    for states in (U, None, U):
        f, c = fresh(), s.coeffs()
        f.set_coeffs(c)
        for q in (s, f):
            q.set_boundary_states(states)
        t1, _ = s.step(3, t=t)
        assert f.step(3, t=t)[0] == t1
        assert np.array_equal(s.coeffs(), f.coeffs())
        assert np.array_equal(s.eval_rhs(c, t=t, dt=0.1), f.eval_rhs(c, t=t, dt=0.1))
        t = t1
        f.close()
    s.close()


def test_adjoint_solves_of_other_lengths_on_one_handle():
    """the kept buffers serve shorter, longer and repeated solves; each equals
    a fresh handle's, and a new mesh starts again"""
    for n in (5, 8):
        mesh = M.structured(n, periodic=False, jitter=0.2, seed=4)
        eps = np.random.default_rng(n).uniform(1.0, 4.0, mesh.K)
        s = None
        for steps, every in ((6, 4), (2, 0), (9, 3), (6, 4)):
            f, _ = make_pair(L.MAXWELL_TE, 2, mesh, eps_elem=eps)
            if s is None:
                s, _ = make_pair(L.MAXWELL_TE, 2, mesh, eps_elem=eps)
            r = []
            for q in (s, f):
                q.project_ic()
                q.set_objective(L.OBJ_PATCH_SQ, (0.1, 0.9, 0.1, 0.9, 2))
                r.append(q.adjoint_solve(steps, 1e-3, every=every, want_eps=True))
            assert r[0][0] == r[1][0] and all(np.array_equal(a, b) for a, b in zip(r[0][1:], r[1][1:]))
            # the objective's sum on the device against the host's
            c, w = s.coeffs(), np.random.default_rng(2).standard_normal(s.shape)
            s.set_objective(L.OBJ_LINEAR, weights=w)
            assert abs(s.objective() - np.vdot(w, c)) <= 1e-13 * np.abs(w * c).sum()
            f.close()
        s.set_mesh(M.structured(n + 1, periodic=False, jitter=0.2, seed=4)).project_ic()
        s.set_objective(L.OBJ_PATCH_SQ, (0.1, 0.9, 0.1, 0.9, 2))
        assert np.isfinite(s.adjoint_solve(3, 1e-3)[1]).all()
        s.close()


def test_ensemble_coefficients_on_the_device():
    """an instance's rows go to and from a device array in one launch (sizes
    around the 256-thread blocks and an odd 8-byte offset), as through the host"""
    import torch
    from dgcuda_amd.ensemble import Ensemble
    E = Ensemble(physics=L.SWE, flux=L.FLUX_ROE, g=9.81, integrator=L.SSPRK3,
                 problem=L.PROB_SWE_BUMP)
    for n, p in ((4, 1), (11, 3), (12, 0), (16, 2)):
        E.add(M.structured(n, periodic=False, jitter=0.2, seed=n), p,
              (1.0, 0.1, 0.5, 0.5, 0.1, 1.0))
    E.build()
    before = [E.coeffs(i) for i in range(4)]
    for i in range(4):
        x = np.random.default_rng(i).standard_normal(before[i].shape)
        d = torch.zeros(2 * x.size + 1, dtype=torch.float64, device="cuda")
        d[1:x.size + 1] = torch.from_numpy(x).reshape(-1).cuda()
        torch.cuda.synchronize()
        a = d.data_ptr() + 8
        assert E.lib.dg_ens_set_coeffs(E.e, i, ctypes.c_void_p(a), L.DEVICE) == 0
        assert np.array_equal(E.coeffs(i), x)
        a += 8 * x.size
        assert E.lib.dg_ens_get_coeffs(E.e, i, ctypes.c_void_p(a), L.DEVICE) == 0
        assert np.array_equal(d[1 + x.size:].cpu().numpy(), x.reshape(-1)) and d[0].item() == 0.0
        for j in range(i + 1, 4):
            assert np.array_equal(E.coeffs(j), before[j])
