"""ThermalLBM.run(n) against n single steps (populations, T, T_old, the heat
source and the stability count, bit for bit) and its statistics against numpy,
at sizes around a block and a wave of the kernels."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd.thermal import ThermalLBM

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (7, 5, 3), (64, 2, 2), (33, 31, 2), (16, 17, 19), (65, 40, 21)]


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
