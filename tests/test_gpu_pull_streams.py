"""The particle-field step of the compact layout where it pulls its populations
past the cache: a duct made of copies of a short one, which stays in the cache,
steps like the short one in every copy, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd import _lib as L
from pourover_amd.engine import HipContext, SolverConfig
from pourover_amd.geometry import link_flags

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shell", [True, False])  # runs off and on the x faces
@pytest.mark.parametrize("precision,shape", [("f32", (112, 128, 52)), ("f32", (149, 101, 47)), ("f64", (101, 97, 36))])
def test_copies_step_alike(precision, shape, shell):
    nx, ny, nz = shape
    copies = 4
    print("case: %d copies of a duct %s %s shell=%s" % (copies, shape, precision, shell), flush=True)
    rng = np.random.default_rng(nx)
    kind = np.zeros((nz, ny, nx), dtype=np.uint8)
    kind[rng.random(kind.shape) < 0.01] = L.POL_KIND_SOLID
    if shell:
        kind[:, (0, -1), :] = L.POL_KIND_SOLID
        kind[:, :, (0, -1)] = L.POL_KIND_SOLID
    periodic = (False, False, True)
    ctx = []
    for n in (1, copies):
        flags, _ = link_flags(np.tile(kind, (n, 1, 1)), periodic=periodic)
        ctx.append(HipContext(SolverConfig(nx, ny, nz * n, precision=precision, les=True, periodic=periodic,
                                           particle_field=True), flags))
    small, large = ctx
    cells, real = int((kind == 0).sum()) * copies, small.pdrag.element_size()
    assert small.layout is not None and (19 + 8) * real * cells > 256 << 20 >= 8 * real * cells
    assert 2 * 19 * real * small.layout.stored_cells <= 256 << 20
    g = torch.Generator(device="cuda").manual_seed(nx)
    rho = 1.0 + 0.02 * (torch.rand((nz, ny, nx), generator=g, device="cuda") - 0.5)
    u = 0.05 * (torch.rand((3, nz, ny, nx), generator=g, device="cuda") - 0.5)
    drag = 1e-3 * torch.rand((4, nz, ny, nx), generator=g, device="cuda")
    drag[:3] *= 0.05
    small.init_equilibrium(rho, u)
    large.init_equilibrium(rho.repeat(copies, 1, 1), u.repeat(1, copies, 1, 1))
    small.pdrag.copy_(drag)
    large.pdrag.copy_(drag.repeat(1, copies, 1, 1))
    for c in ctx:
        c.step(3)
        c.macroscopic(macro=True)
    f, rho, u = small.dense_populations(), small.rho, small.u
    assert torch.isfinite(f).all() and (f != 0).any()
    assert torch.equal(large.dense_populations(), f.repeat(1, copies, 1, 1))
    assert torch.equal(large.rho, rho.repeat(copies, 1, 1)) and torch.equal(large.u, u.repeat(1, copies, 1, 1))
