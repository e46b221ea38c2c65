"""Device arrays whose allocation ends before the array does: refused by every
call that a kernel would reach them from, as a copy refuses them, and before
anything is launched.  The whole allocation is taken."""
import ctypes

import numpy as np
import pytest
import torch  # noqa: F401  (before the library, so that both use one HIP runtime)

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair

pytestmark = pytest.mark.gpu


class _Alloc:
    """an allocation of its own (torch's tensors share larger ones), from the HIP
    runtime that the library is linked to"""

    def __init__(self, nbytes):
        self.hip = L.load()
        self.p = ctypes.c_void_p()
        assert self.hip.hipMalloc(ctypes.byref(self.p), ctypes.c_size_t(nbytes)) == 0
        assert self.hip.hipMemset(self.p, 0, ctypes.c_size_t(nbytes)) == 0
        assert self.hip.hipDeviceSynchronize() == 0

    def at(self, off):
        return ctypes.c_void_p(self.p.value + off)

    def close(self):
        assert self.hip.hipFree(self.p) == 0


def test_short_device_arrays_are_refused():
    mesh = M.structured(60, periodic=False, jitter=0.2, seed=4)
    s, _ = make_pair(L.EULER, 2, mesh)
    s.project_ic()
    sb, half = 8 * s.size, 8 * (s.size // 2)
    a, b, c = _Alloc(sb), _Alloc(sb), _Alloc(sb)
    assert s.lib.dg_get_coeffs(s.h, a.at(0), L.DEVICE) == 0
    assert s.lib.dg_eval_rhs(s.h, a.at(0), 0.0, 1.0, b.at(0), L.DEVICE) == 0
    assert s.lib.dg_adjoint_rhs(s.h, a.at(0), 0.0, 1.0, b.at(0), c.at(0), L.DEVICE) == 0
    bad = half, 0, 0
    for i in range(3):
        x = bad[-i:] + bad[:-i]
        if i < 2:
            print("short rhs", x[:2], flush=True)
            assert s.lib.dg_eval_rhs(s.h, a.at(x[0]), 0.0, 1.0, b.at(x[1]), L.DEVICE) == L.DG_ERR_HIP
            assert b"ends before" in s.lib.dg_last_error(s.h)
        print("short vjp", x, flush=True)
        assert s.lib.dg_adjoint_rhs(s.h, a.at(x[0]), 0.0, 1.0, b.at(x[1]), c.at(x[2]),
                                    L.DEVICE) == L.DG_ERR_HIP
        assert b"ends before" in s.lib.dg_last_error(s.h)
    # the handle goes on as before
    assert s.lib.dg_eval_rhs(s.h, a.at(0), 0.0, 1.0, b.at(0), L.DEVICE) == 0
    for x in (a, b, c):
        x.close()
    s.close()


def test_short_device_arrays_of_an_ensemble_are_refused():
    from dgcuda_amd.ensemble import Ensemble
    E = Ensemble(physics=L.SWE)
    E.add(M.structured(60, periodic=False, jitter=0.2, seed=1), 2, (1.0, 0.1, 0.5, 0.5, 0.1, 1.0))
    E.build(64)
    c = E.coeffs(0)
    a = _Alloc(c.nbytes)
    assert E.lib.dg_ens_get_coeffs(E.e, 0, a.at(0), L.DEVICE) == 0
    for call in (E.lib.dg_ens_get_coeffs, E.lib.dg_ens_set_coeffs):
        print("short", call.__name__, flush=True)
        assert call(E.e, 0, a.at(8 * (c.size // 2)), L.DEVICE) == L.DG_ERR_HIP
        assert b"ends before" in E.lib.dg_ens_last_error(E.e)
    assert E.lib.dg_ens_set_coeffs(E.e, 0, a.at(0), L.DEVICE) == 0
    assert np.array_equal(E.coeffs(0), c)
    a.close()
    E.close()
