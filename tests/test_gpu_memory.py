"""Device memory of the adjoint's calls: what a solve leaves for the next one on
its handle is given back on request, with the handle, with its mesh, and when an
allocation of another handle fails; a product on host data keeps nothing."""
import gc

import numpy as np
import pytest
import torch

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair

pytestmark = pytest.mark.gpu

MiB = 1 << 20


def _free():
    gc.collect()
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _solver(n=120):
    mesh = M.structured(n, periodic=False, jitter=0.2, seed=4)
    eps = np.random.default_rng(3).uniform(1.0, 4.0, mesh.K)
    s, _ = make_pair(L.MAXWELL_TE, 3, mesh, eps_elem=eps)
    s.project_ic()
    s.set_objective(L.OBJ_PATCH_SQ, (0.1, 0.9, 0.1, 0.9, 2))
    return s


def _solve(s, steps=16, every=16):
    s.project_ic()
    return s.adjoint_solve(steps, 1e-4, every=every, want_eps=True)


def test_buffers_left_by_a_solve_are_given_back():
    s, o = _solver(), _solver(4)  # a state is 6.9 MB, a solve of 16 steps 0.75 GB
    for q in (s, o):
        q.step(2, dt=1e-4)
        _solve(q, 2, 1)  # code, streams and the kernels' scratch are in place
        q.eval_rhs(q.coeffs())
        q.adjoint_release()
    before = _free()
    want = _solve(s)
    kept = before - _free()
    print("kept", kept // MiB, "MiB", flush=True)
    assert kept > 256 * MiB  # (else nothing is tested here)
    s.adjoint_release()
    s.adjoint_release()
    assert before - _free() < 8 * MiB
    # a solve after the release, a shorter one in the longer one's buffers
    for steps, every in ((16, 16), (4, 2), (16, 16)):
        got = _solve(s, steps, every)
    assert got[0] == want[0] and all(np.array_equal(a, b) for a, b in zip(got[1:], want[1:]))
    # another handle's allocation that fails takes them, and says so itself
    assert before - _free() > 256 * MiB
    with pytest.raises(L.DgError, match="hipMalloc of .* bytes failed"):
        o.adjoint_solve(10 ** 9, 1e-4, every=10 ** 9)  # 10 TB and more
    assert before - _free() < 64 * MiB
    # both go on
    assert np.isfinite(o.eval_rhs(o.coeffs())).all()
    assert np.array_equal(_solve(s)[1], want[1])
    # a new mesh, then the end of the handle
    s.set_mesh(M.structured(4, periodic=False, jitter=0.2, seed=4))
    assert before - _free() < 64 * MiB
    o.close()
    s.close()
    s = _solver()
    at = _free()
    _solve(s)
    s.close()
    assert _free() > at
    s.close()


def test_host_products_keep_no_array():
    mesh = M.structured(160, periodic=False, jitter=0.2, seed=4)
    held = []
    for product in (False, True):
        s, _ = make_pair(L.EULER, 3, mesh)
        s.project_ic()
        u = s.coeffs()
        s.eval_rhs(u)
        if held:
            s.adjoint_rhs(u, u)
        before = _free()
        s.close()
        held.append(_free() - before)
        print("product", product, "freed with the handle", held, "state", u.nbytes, flush=True)
        if not product:
            s, _ = make_pair(L.EULER, 3, mesh)  # code in place before the second round
            s.project_ic()
            s.adjoint_rhs(u, u)
            s.close()
    assert abs(held[1] - held[0]) < u.nbytes // 2
