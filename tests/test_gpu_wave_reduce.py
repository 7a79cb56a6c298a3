"""The wave reductions (wave_reduce: DPP moves and half-row / half-wave swaps)
see every lane once: a field that differs from a uniform one in a single cell
changes the sums, counts and extremes of pol_field_stats and pol_reduce by that
cell's share, wherever in its wave the cell lies."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd import diagnostics as D
from pourover_amd.engine import HipContext, SolverConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 4, 2), (35, 3, 2)])  # 4-cell loads; one cell a lane
def test_field_statistics_see_every_lane(shape):
    nx, ny, nz = shape
    ctx = HipContext(SolverConfig(nx, ny, nz))
    for i in range(nx * ny):
        ctx.rho.fill_(1.0)
        ctx.u.zero_()
        ctx.rho.view(-1)[i] = 1.5
        ctx.u.view(3, -1)[:, i] = torch.tensor([0.25, -0.5, 0.0])
        s, zp = D.field_statistics(ctx)
        assert s["cells"] == nx * ny * nz and s["sum_drho"] == 0.5 and s["max_abs_drho"] == 0.5, i
        assert s["mom_x"] == 0.375 and s["mom_y"] == -0.75 and s["sum_ux2"] == 0.0625, i
        assert s["umag_active"] == 1 and s["fluid_rho_max"] == 1.5 and s["fluid_rho_min"] == 1.0, i
        assert s["max_umag"] == float(np.sqrt(np.float32(0.3125))) and s["sum_umag"] == s["max_umag"], i
        assert zp[0] == nx * ny + 0.5 and zp[1] == nx * ny


def test_reduction_sees_every_lane():
    ctx = HipContext(SolverConfig(16, 8, 4, precision="f64"))
    n = 512
    for i in range(256):
        # a rest population of D_0 = 18 more: rho = 1.5 in one cell
        ctx.f_current.zero_()
        ctx.f_current[0, i] = 18.0
        d = ctx.reduce()
        assert d["mass"] == n + 0.5 and d["rho_max"] == 1.5 and d["rho_min"] == 1.0 and d["cells"] == n, i
