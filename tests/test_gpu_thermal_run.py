"""ThermalLBM.run(n) against n single steps (populations, T, T_old, the heat
source and the stability count, bit for bit) and its statistics against numpy,
at sizes around a block and a wave of the kernels."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import thermal as OT
from pourover_amd.thermal import ThermalFluidCoupledSolver, ThermalLBM

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (7, 5, 3), (64, 2, 2), (33, 31, 2), (16, 17, 19), (65, 40, 21), (70, 66, 60)]


def _make(shape, precision, convection, seed=3):
    th = ThermalLBM(grid=shape, precision=precision)
    rng = np.random.default_rng(seed)
    th.initialize_from(rng.uniform(20.0, 90.0, shape))
    th.enable_convection_coupling(convection)
    if convection:
        u = torch.from_numpy(rng.uniform(-0.02, 0.02, tuple(th._vel.shape))).to(th._vel)
        th.set_velocity_field(u)
    return th


@pytest.mark.parametrize("convection", [False, True])
@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_run_equals_single_steps(shape, precision, convection):
    for n in (1, 2, 3, 4):
        print("case: thermal run(%d) %s %s convection=%s" % (n, shape, precision, convection), flush=True)
        a, b = _make(shape, precision, convection), _make(shape, precision, convection)
        # a boundary temperature that is not the sum of the populations: a
        # run leaves it readable as T_old of its first step
        mask = np.zeros(shape, np.uint8)
        mask[0] = 1
        for th in (a, b):
            th.apply_dirichlet_bc(mask, 90.1)
        ok = a.run(n)
        ok1 = [b.step() for _ in range(n)][-1]
        assert ok == ok1
        for name in ("temperature", "temperature_old", "heat_source"):
            assert torch.equal(getattr(a, name).to_torch(), getattr(b, name).to_torch()), name
        assert torch.equal(a.g_device, b.g_device)


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_step_with_velocity(shape, precision):
    """The velocity handed over inside the step: the state and the velocity
    buffer of set_velocity_field and step, for a device velocity, one that
    needs a conversion or a copy, and the solver's own buffer."""
    rng = np.random.default_rng(11)
    a, b = _make(shape, precision, True), _make(shape, precision, True)
    other = torch.float64 if precision == "f32" else torch.float32
    for kind in ("same", "type", "strided", "own", "host"):
        u = torch.from_numpy(rng.uniform(-0.02, 0.02, tuple(a._vel.shape))).to(a._vel)
        u = {"same": u, "type": u.to(other), "strided": u.flip(0).transpose(1, 3).contiguous().transpose(1, 3),
             "own": None, "host": u.cpu()}[kind]
        ok = a.step_with_velocity(a._vel if u is None else u)
        b.set_velocity_field(b._vel if u is None else u)
        assert ok == b.step()
        for x, y in ((a._vel, b._vel), (a.g_device, b.g_device), (a._hs, b._hs), (a._T[a._tcur], b._T[b._tcur])):
            assert torch.equal(x, y), kind


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES + [(128, 64, 33), (101, 103, 107)])
def test_statistics(shape, precision):
    print("case: thermal statistics %s %s" % (shape, precision), flush=True)
    th = _make(shape, precision, True)
    T = th.temperature.to_torch().double().cpu().numpy()
    n, eps = T.size, np.finfo(np.float64).eps
    lo, hi, mean = th.get_temperature_stats()
    assert lo == T.min() and hi == T.max()
    assert abs(mean * n - T.sum()) <= n * eps * np.abs(T).sum() + 2 * eps * abs(mean * n)  # any order of the sum
    coupled = ThermalFluidCoupledSolver(fluid_solver=_Fluid(), thermal_solver=th)
    assert coupled._check_coupling_stability()
    for at in (0, n // 2, n - 1):  # |u| > 1 in one cell, wherever it lies
        th._vel.view(3, -1)[:, at] = torch.tensor([0.6, 0.6, -0.6])
        assert not coupled._check_coupling_stability()
        th._vel.view(3, -1)[:, at] = torch.tensor([float("nan"), 2.0, 0.0])  # as a norm of NaN: not above 1
        assert coupled._check_coupling_stability()
        th._vel.view(3, -1)[:, at] = torch.tensor([float("inf"), 0.0, 0.0])
        assert not coupled._check_coupling_stability()
        th._vel.view(3, -1)[:, at] = 0.0
    th.temperature.to_torch().view(-1)[n - 1] = 151.0
    assert not coupled._check_coupling_stability()
    th.temperature.to_torch().view(-1)[n - 1] = -11.0
    assert not coupled._check_coupling_stability()


@pytest.mark.parametrize("shape", SHAPES)
def test_count_of_unstable_cells(shape):
    """0, 1, some and all cells outside the stability bounds, and afresh after each."""
    n = shape[0] * shape[1] * shape[2]
    for share in (0.0, 0.3, 1.0, 0.0):
        th = _make(shape, "f32", False)
        rng = np.random.default_rng(int(share * 10))
        T = np.where(rng.random(shape) < share, np.float32(1e4), np.float32(50.0))
        th.initialize_from(T)
        ok = th.step()
        g = th.g_device.cpu().numpy()
        Tn = th.temperature.to_torch().cpu().numpy()
        bad = (Tn < -50) | (Tn > 150) | (np.abs(g) > 1000).any(axis=0)
        assert th._last_unstable == int(bad.sum()) and ok == (not bad.any())
    assert n > 0


class _Fluid:
    """The coupled solver asks its fluid solver for nothing in these checks."""


@pytest.mark.parametrize("convection", [False, True])
@pytest.mark.parametrize("precision,shape", [("f32", (171, 168, 173)), ("f64", (131, 130, 145))])
def test_streaming_steps(precision, shape, convection):
    """Population buffers above the last-level cache (stores past the cache):
    three steps in one run and one by one against the numpy restatement."""
    print("case: streaming thermal steps %s %s convection=%s" % (shape, precision, convection), flush=True)
    a = _make(shape, precision, convection)
    assert 2 * a.g_device.numel() * a.g_device.element_size() > 256 << 20
    T = np.ascontiguousarray(a.temperature.to_numpy())
    st = {"g": OT.equilibrium(T), "T": T, "heat_source": np.zeros_like(T),
          "u": np.ascontiguousarray(a._vel.cpu().numpy().transpose(3, 2, 1, 0))}
    assert a.run(3)
    for _ in range(3):
        st = OT.step(st, a.omega_thermal, convection=convection)
    assert np.array_equal(a.g, st["g"]) and np.array_equal(a.temperature.to_numpy(), st["T"])
    assert np.array_equal(a.temperature_old.to_numpy(), st["T_old"])
    assert np.array_equal(a.heat_source.to_numpy(), st["heat_source"])


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES + [(128, 64, 33), (101, 103, 107)])
def test_statistics_of_the_step(shape, precision):
    """A step's own coupling statistics: those of the pass over its result, and
    afresh after a step with fast cells (|u| just at, next to and above 1)."""
    print("case: statistics of the step %s %s" % (shape, precision), flush=True)
    th = _make(shape, precision, True)
    n, eps = th._hs.numel(), np.finfo(np.float64).eps
    rng = np.random.default_rng(17)
    one = th._hs.new_ones(1)
    after = torch.nextafter(one, 2 * one)  # a square of it is above one, its root rounds to it
    for speeds in ([], [one, -one], [after], [3 * one, float("nan") * one, float("inf") * one], []):
        u = torch.from_numpy(rng.uniform(-0.02, 0.02, tuple(th._vel.shape))).to(th._vel)
        cells = rng.choice(n, len(speeds), replace=False)
        for c, v in zip(cells, speeds):
            u.view(3, -1)[:, c] = 0.0
            u.view(3, -1)[rng.integers(3), c] = v
        got, want = np.zeros(4), np.zeros(4)
        th.initialize_from(rng.uniform(20.0, 90.0, shape))
        ok = th.step_with_velocity(u, got)
        th._coupling_stats(want)
        uu = u.view(3, -1).cpu().numpy()
        assert want[3] == (np.sqrt((uu[0] * uu[0] + uu[1] * uu[1]) + uu[2] * uu[2]) > 1).sum()
        T = th.temperature.to_torch().double().cpu().numpy()
        bad = (th.g_device.isnan() | (th.g_device.abs() > 1000)).any(dim=0).cpu().numpy() | ~((T >= -50) & (T <= 150))
        assert th._last_unstable == int(bad.sum()) and ok == (not bad.any())
        assert np.array_equal(got[[0, 1, 3]], want[[0, 1, 3]])
        if np.isfinite(T).all():
            assert abs(got[2] - want[2]) <= 2 * n * eps * np.abs(T).sum()  # any order of the sum


@pytest.mark.parametrize("precision,shape", [("f32", (171, 168, 173)), ("f32", (171, 167, 175)), ("f64", (131, 130, 145)),
                                             ("f64", (131, 131, 145))])
def test_streaming_step_with_velocity(precision, shape):
    """The hand-over and the statistics of a step past the cache, in cell counts
    that are and are not a multiple of four."""
    print("case: streaming step with velocity %s %s" % (shape, precision), flush=True)
    a, b = _make(shape, precision, True), _make(shape, precision, True)
    assert 2 * a.g_device.numel() * a.g_device.element_size() > 256 << 20
    u = torch.from_numpy(np.random.default_rng(11).uniform(-0.02, 0.02, tuple(a._vel.shape))).to(a._vel)
    u.view(3, -1)[0, -3:] = 1.5
    for th in (a, b):
        th.use_base_heat_source(torch.full_like(th._hs, 1e-3))
    got, want = np.zeros(4), np.zeros(4)
    ok = a.step_with_velocity(u, got)
    b.set_velocity_field(u)
    assert ok and b.step()
    for x, y in ((a._vel, b._vel), (a.g_device, b.g_device), (a._hs, b._hs), (a._T[a._tcur], b._T[b._tcur])):
        assert torch.equal(x, y)
    b._coupling_stats(want)
    assert np.array_equal(got[[0, 1, 3]], want[[0, 1, 3]]) and got[3] == 3
    n, eps = b._hs.numel(), np.finfo(np.float64).eps
    assert abs(got[2] - want[2]) <= 2 * n * eps * abs(want[2])  # positive terms, any order
