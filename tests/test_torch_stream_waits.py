"""The solver's stream does not wait for torch's: before every call that reads
or writes a CUDA tensor, Solver has waited for what torch queued on its current
stream.  On stand-ins for torch, the library and the tensors (the race itself
would need luck to show): each call finds the stream waited for, whichever side
its tensors are on."""
import types

import numpy as np
import pytest

from dgcuda_amd import _lib as L
from dgcuda_amd import solver as S

SHAPE = (1, 3, 2)
SIZE = 6


class FakeTensor:
    dtype = "f64"

    def __init__(self, world, shape=SHAPE):
        self.world, self.shape = world, shape
        self.device = types.SimpleNamespace(type="cuda", index=0)
        world.pending = True  # torch has queued work on the tensor's memory

    def numel(self):
        return int(np.prod(self.shape))

    def is_contiguous(self):
        return True

    def contiguous(self):
        return self

    def data_ptr(self):
        return 4096


FakeTensor.__module__ = "torch"


class World:
    """torch and the library: `pending` is unfinished work on torch's stream"""
    pending = False
    capturing = False
    calls = ()
    float64 = "f64"

    def __init__(self):
        self.calls = []
        stream = types.SimpleNamespace(synchronize=self._synchronize)
        self.cuda = types.SimpleNamespace(is_current_stream_capturing=lambda: self.capturing,
                                          current_stream=lambda device: stream)

    def _synchronize(self):
        self.pending = False
        self.calls.append("wait")

    def empty(self, shape, dtype, device):
        # (queues nothing itself: the memory's last use may still be pending)
        was = self.pending
        t = FakeTensor(self, shape if isinstance(shape, tuple) else (shape,))
        self.pending = was
        return t

    def __getattr__(self, name):
        if not name.startswith("dg_"):
            raise AttributeError(name)

        def call(*a):
            if name not in ("dg_info", "dg_last_error"):
                assert not self.pending, "%s before torch's stream was waited for" % name
                self.calls.append(name)
            return 0
        return call


@pytest.fixture
def world(monkeypatch):
    w = World()
    monkeypatch.setattr(S, "_torch", lambda: w)
    return w


@pytest.fixture
def solver(world):
    s = S.Solver.__new__(S.Solver)
    s.lib, s.h, s.cfg = world, None, types.SimpleNamespace(device=0)
    s.physics, s.p, s.N, s.n_p, s.K = L.ADVECTION, 1, 1, 3, 2
    return s


@pytest.mark.parametrize("call,name", [
    (lambda s, w: s.set_coeffs(FakeTensor(w)), "dg_set_coeffs"),
    (lambda s, w: s.coeffs(out=FakeTensor(w)), "dg_get_coeffs"),
    (lambda s, w: s.eval_rhs(FakeTensor(w), out=FakeTensor(w)), "dg_eval_rhs"),
    (lambda s, w: s.eval_rhs(FakeTensor(w)), "dg_eval_rhs"),
    (lambda s, w: s.adjoint_rhs(FakeTensor(w), FakeTensor(w)), "dg_adjoint_rhs"),
    (lambda s, w: s.set_objective(L.OBJ_LINEAR, weights=FakeTensor(w)), "dg_adjoint_set_objective"),
    (lambda s, w: s.adjoint_solve(2, 0.1, device="cuda"), "dg_adjoint_solve"),
    (lambda s, w: s.adjoint_solve(2, 0.1, want_eps=True, device="cuda"), "dg_adjoint_solve")])
def test_calls_wait_for_torchs_stream(solver, world, call, name):
    world.pending = True
    call(solver, world)
    assert name in world.calls and world.calls[0] == "wait"


def test_host_arrays_wait_for_nothing(solver, world):
    u = np.zeros(SHAPE)
    solver.set_coeffs(u)
    solver.coeffs()
    solver.eval_rhs(u)
    solver.adjoint_rhs(u, u)
    solver.adjoint_solve(2, 0.1)
    assert "wait" not in world.calls


def test_no_wait_while_torch_captures(solver, world):
    world.capturing = True
    t = FakeTensor(world)
    world.pending = False
    solver.set_coeffs(t)
    assert world.calls == ["dg_set_coeffs"]
