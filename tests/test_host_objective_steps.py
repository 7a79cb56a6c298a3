"""The recorded forward run of AdjointProblem asks objective_step() which steps
count, as the step-by-step run does, also where a subclass has its own.
Without a device: the library is a recorder whose flux of step n is 2^n."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from pourover_amd import adjoint as A


class _Lib:
    def __init__(self):
        self.steps = []  # (count, flux_first) of every recorded run
        self.at = 0

    def pol_step_record(self, handle, states, stride, count, final, first, flux, stream):
        self.steps.append((count, first))
        if first < count:
            out = np.ctypeslib.as_array(C.cast(flux, C.POINTER(C.c_double)), (count - first,))
            out[:] = [2.0 ** (self.at + i) for i in range(first, count)]
        return 0


class _Ctx:
    handle, current = None, 0

    def __init__(self):
        self.lib = _Lib()
        self.f_current, self.f_next = torch.zeros(4), torch.zeros(4)

    def set_current(self, i):
        self.current = i

    def init_equilibrium(self):
        self.lib.at = 0

    def step(self, n, what=0):
        assert n == 1
        red = np.zeros(12)
        red[7] = 2.0 ** self.lib.at
        self.lib.at += 1
        return red if what else None


def _problem(cls, steps, window, checkpoint):
    p = object.__new__(cls)
    p.ctx, p.steps, p.window = _Ctx(), steps, window
    p.store_all = checkpoint is None
    p.checkpoint = steps if p.store_all else checkpoint
    p.seg = torch.zeros((p.checkpoint, 4))
    p.ckpt = None if p.store_all else torch.zeros((steps // p.checkpoint, 4))
    return p


class _EveryThird(A.AdjointProblem):
    def objective_step(self, n):
        return n % 3 == 1


@pytest.mark.parametrize("cls", [A.AdjointProblem, _EveryThird])
@pytest.mark.parametrize("checkpoint", [None, 1, 4, 12])
@pytest.mark.parametrize("window", [0, 1, 5, 12, 20])
def test_the_recorded_run_counts_the_objective_steps(monkeypatch, cls, checkpoint, window):
    monkeypatch.setattr(A.L, "stream_handle", lambda stream=None: None)
    p = _problem(cls, 12, window, checkpoint)
    want = sum(2.0 ** n for n in range(12) if p.objective_step(n))
    assert p.forward(checkpoints=False) == want
    assert p.forward(checkpoints=True) == want
    (count, first), = p.ctx.lib.steps
    assert count == p.checkpoint and 0 <= first <= count
    if cls is A.AdjointProblem:  # nothing is reduced before the window
        assert first == min(count, max(0, (12 - window) - (12 - count)))
