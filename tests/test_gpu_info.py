"""dg_info names the registers of the stage kernel in use: the point-parallel
one's on small meshes, the large meshes' above.  The two differ by far at the
orders here: a thread per element holds its state and accumulators (p = 3,
Euler: 80 doubles, 160 registers, and more), a thread per point does not."""
import pytest

from dgcuda_amd import _lib as L
from dgcuda_amd import mesh as M
from tests.helpers import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics,p,big", [(L.EULER, 2, 92), (L.EULER, 3, 86),
                                           (L.MAXWELL_TE, 3, 93)])
def test_registers_of_the_stage_in_use(physics, p, big):
    s, _ = make_pair(physics, p, M.structured(4, periodic=False, jitter=0.2, seed=1))
    small = s.info().vgprs_stage
    s.set_mesh(M.structured(big, periodic=False, jitter=0.2, seed=1))
    wide = s.info().vgprs_stage
    s.set_mesh(M.structured(5, periodic=False, jitter=0.2, seed=1))
    print("physics", physics, "p", p, "small", small, "wide", wide, flush=True)
    assert s.info().vgprs_stage == small and 0 < small < wide <= 512
    s.close()
