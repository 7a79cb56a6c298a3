"""The FP64 reductions' fold over the blocks (k_reduce_fold): block counts at
the edges of its one- and two-launch forms, against float64 sums of the rho / u
fields of the same state (FP64 storage: the fields hold the reduced values)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd.engine import HipContext, SolverConfig

pytestmark = pytest.mark.gpu


# blocks of 256 cells: 1, 2, 21 + 1 rows, 512 (one launch), 513, 514 and 1024 (two launches)
@pytest.mark.parametrize("shape", [(2, 2, 2), (129, 2, 2), (32, 16, 11), (64, 64, 32), (3, 4, 10923), (113, 97, 12),
                                   (64, 64, 64)])
def test_reductions_match_field_sums(shape):
    nx, ny, nz = shape
    print("case: reduction fold %s" % (shape,), flush=True)
    ctx = HipContext(SolverConfig(nx, ny, nz, precision="f64"))
    g = torch.Generator().manual_seed(nx + 7 * ny)
    rho = 1.0 + 0.1 * (torch.rand((nz, ny, nx), generator=g, dtype=torch.float64) - 0.5)
    u = 0.1 * (torch.rand((3, nz, ny, nx), generator=g, dtype=torch.float64) - 0.5)
    ctx.init_equilibrium(rho, u)
    d = ctx.reduce()
    ctx.macroscopic(macro=True)
    r, v = ctx.rho.cpu().numpy().ravel(), ctx.u.cpu().numpy().reshape(3, -1)
    n, eps = r.size, np.finfo(np.float64).eps
    usq = v[0] * v[0] + v[1] * v[1] + v[2] * v[2]
    # each sum is off by at most n eps times the sum of magnitudes in any order
    for key, x in (("mass", r), ("mom_x", r * v[0]), ("mom_y", r * v[1]), ("mom_z", r * v[2]),
                   ("kinetic_energy", 0.5 * r * usq)):
        assert abs(d[key] - x.sum()) <= n * eps * np.abs(x).sum() + 1e-300, key
    assert d["cells"] == n and d["nonfinite_cells"] == 0
    assert d["rho_min"] == r.min() and d["rho_max"] == r.max()
    assert abs(d["max_velocity"] - np.sqrt(usq.max())) <= 4 * eps * d["max_velocity"]
    assert ctx.reduce() == d  # a fixed order: the same bits again
