"""ThermalFluidCoupledSolver calls the methods of the thermal solver that a
caller hands it (thermal_fluid_coupled.py:143-262): its own step,
set_velocity_field, get_temperature_stats and compute_diagnostics, from a
subclass, replaced on the object or the class, or of an object that has only
those; the native step that does their work in one call serves the package's
own.  Without a device: the library is a recorder."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd import thermal as TH

SHAPE = (3, 4, 5)  # nz, ny, nx
MODES = ["subclass", "object", "class"]


class _Lib:
    """Every native call: recorded, succeeds; statistics are zeros."""

    def __init__(self, calls):
        self.calls = calls

    def __getattr__(self, name):
        def call(*a):
            self.calls.append(name)
            return 0
        return call


class _Fluid:
    def __init__(self, calls):
        self.calls = calls
        self.u = torch.full((3,) + SHAPE, 0.25)

    def init_fields(self):
        pass

    def step(self):
        self.calls.append("fluid")


class _Handle:
    handle = None


def _thermal(calls, cls=None):
    """A ThermalLBM whose buffers are on the host and whose library records."""
    th = object.__new__(cls or TH.ThermalLBM)
    th.lib, th.ctx = _Lib(calls), _Handle()
    th.nz, th.ny, th.nx = SHAPE
    th._vel, th._hs, th._hs_base = torch.zeros((3,) + SHAPE), torch.zeros(SHAPE), torch.zeros(SHAPE)
    th._gcur = th._tcur = th.current_step = th._last_unstable = 0
    th.omega_thermal = 1.0
    th.reset_source_each_step = False
    th.is_initialized = True
    th.enable_convection = False
    return th


def _coupled(monkeypatch, calls, th, **config):
    monkeypatch.setattr(TH.L, "stream_handle", lambda stream=None: None)
    s = TH.ThermalFluidCoupledSolver(TH.CouplingConfig(**config), fluid_solver=_Fluid(calls), thermal_solver=th)
    s.is_initialized = True
    calls.clear()
    return s


@pytest.mark.parametrize("subcycles", [0, 1, 3])
def test_the_packages_own_solver_takes_one_native_call(monkeypatch, subcycles):
    calls = []
    s = _coupled(monkeypatch, calls, _thermal(calls), thermal_subcycles=subcycles)
    assert s.step()
    later = ["pol_thermal_step"] * (subcycles - 1)
    stats = [] if subcycles == 1 else ["pol_thermal_coupling_stats"]
    assert calls == ["fluid"] + (["pol_thermal_step_with_velocity"] if subcycles else []) + later + stats


def _replace(monkeypatch, calls, mode, name, fn):
    if mode == "subclass":
        return _thermal(calls, type("Own", (TH.ThermalLBM,), {name: fn}))
    if mode == "class":
        monkeypatch.setattr(TH.ThermalLBM, name, fn)
        return _thermal(calls)
    th = _thermal(calls)
    monkeypatch.setattr(th, name, fn.__get__(th), raising=False)
    return th


@pytest.mark.parametrize("subcycles", [1, 2])
@pytest.mark.parametrize("mode", MODES)
def test_an_own_step_runs_every_sub_cycle(monkeypatch, mode, subcycles):
    calls = []

    def step(self):
        calls.append("own step")
        assert torch.equal(self._vel, torch.full_like(self._vel, 0.25))  # handed over before
        return True

    s = _coupled(monkeypatch, calls, _replace(monkeypatch, calls, mode, "step", step), thermal_subcycles=subcycles)
    assert s.step()
    assert calls == ["fluid"] + ["own step"] * subcycles + ["pol_thermal_coupling_stats"]


@pytest.mark.parametrize("mode", MODES)
def test_an_own_set_velocity_field_takes_the_velocity(monkeypatch, mode):
    calls = []

    def set_velocity_field(self, velocity_field):
        calls.append("own velocity")
        self._vel.copy_(velocity_field * 0.5)  # say, smoothed

    th = _replace(monkeypatch, calls, mode, "set_velocity_field", set_velocity_field)
    s = _coupled(monkeypatch, calls, th)
    assert s.step()
    assert calls == ["fluid", "own velocity", "pol_thermal_step", "pol_thermal_coupling_stats"]
    assert torch.equal(th._vel, torch.full_like(th._vel, 0.125))


@pytest.mark.parametrize("name", ["get_temperature_stats", "compute_diagnostics"])
@pytest.mark.parametrize("mode", MODES)
def test_own_statistics_decide_the_stability(monkeypatch, mode, name):
    calls, stats = [], [20.0, 90.0, 50.0]

    def own(self):
        calls.append("own statistics")
        return tuple(stats)

    th = _replace(monkeypatch, calls, mode, name, own)
    s = _coupled(monkeypatch, calls, th)
    assert s.step() and calls == ["fluid", "pol_thermal_step_with_velocity", "own statistics"]
    stats[1] = 151.0
    assert not s.step()
    stats[1] = 90.0
    assert s.step()
    th._vel[0, 1, 1, 1] = 1.5  # the recorder leaves the velocity buffer alone
    assert not s.step()


@pytest.mark.parametrize("subcycles", [0, 1, 2])
def test_an_object_with_the_documented_methods_only(monkeypatch, subcycles):
    calls = []

    class Plain:
        _hs, _vel = torch.zeros(SHAPE), torch.zeros((3,) + SHAPE)

        def enable_convection_coupling(self, enable):
            pass

        def use_base_heat_source(self, base):
            pass

        def reset_heat_source_to_base(self, base):
            calls.append("reset")

        def set_velocity_field(self, v):
            calls.append("velocity")

        def step(self):
            calls.append("step")
            return True

        def get_temperature_stats(self):
            calls.append("statistics")
            return np.float32(20), np.float32(90), np.float32(50)

    s = _coupled(monkeypatch, calls, Plain(), thermal_subcycles=subcycles)
    assert s.step()
    assert calls == ["fluid", "velocity"] + ["reset"] * (subcycles != 1) + ["step"] * subcycles + ["statistics"]


def test_no_velocity_is_refused(monkeypatch):
    calls = []
    s = _coupled(monkeypatch, calls, _thermal(calls))
    s.fluid_solver.u = None
    with pytest.raises(TypeError):
        s.step()


@pytest.mark.parametrize("subcycles", [0, 1, 2])
@pytest.mark.parametrize("mode", MODES)
def test_an_own_stability_check_takes_no_argument(monkeypatch, mode, subcycles):
    """_check_coupling_stability is the reference's own name (thermal_fluid_coupled.py:237)."""
    calls, answer = [], [True]

    def check(self):
        calls.append("own check")
        return answer[0]

    cls = TH.ThermalFluidCoupledSolver
    if mode == "subclass":
        monkeypatch.setattr(TH, "ThermalFluidCoupledSolver", type("Own", (cls,), {"_check_coupling_stability": check}))
    elif mode == "class":
        monkeypatch.setattr(cls, "_check_coupling_stability", check)
    s = _coupled(monkeypatch, calls, _thermal(calls), thermal_subcycles=subcycles)
    if mode == "object":
        monkeypatch.setattr(s, "_check_coupling_stability", check.__get__(s))
    assert s.step() and calls[-1] == "own check" and calls.count("own check") == 1
    answer[0] = False
    assert not s.step()


def test_a_velocity_that_the_step_would_overwrite_is_copied_first(monkeypatch):
    calls = []
    th = _thermal(calls)
    s = _coupled(monkeypatch, calls, th)
    lib = th.lib
    th.lib = type("Refuses", (), {
        "pol_thermal_step_with_velocity": staticmethod(lambda *a: TH.L.POL_ERR_INVALID),
        "__getattr__": lambda self, name: getattr(lib, name)})()
    assert s.step()
    assert torch.equal(th._vel, torch.full_like(th._vel, 0.25))
    assert calls == ["fluid", "pol_thermal_step", "pol_thermal_coupling_stats"]
