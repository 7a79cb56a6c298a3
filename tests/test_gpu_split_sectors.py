"""Dense boxes above the last-level cache whose population planes are no whole
number of 64-byte sectors apart (cached stores, groups of 32 blocks per XCD)
and ones whose planes are (streaming stores): a periodic box made of copies of
a small one, which stays in the cache, steps like the small one in every copy,
bit for bit."""
from __future__ import annotations

import pytest
import torch

from pourover_amd.engine import HipContext, SolverConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("les", [False, True])  # the plain and the general kernel
@pytest.mark.parametrize("precision,shape,copies", [("f32", (131, 127, 27), 4), ("f32", (112, 128, 32), 4),
                                                    ("f16", (211, 131, 33), 4), ("bf16", (241, 127, 24), 5),
                                                    ("f64", (101, 97, 23), 4)])
def test_copies_step_alike(precision, shape, copies, les):
    nx, ny, nz = shape
    print("case: %d copies of %s %s les=%s" % (copies, shape, precision, les), flush=True)
    small = HipContext(SolverConfig(nx, ny, nz, precision=precision, les=les))
    large = HipContext(SolverConfig(nx, ny, nz * copies, precision=precision, les=les))
    size = 2 * large.f[0].numel() * large.f[0].element_size()
    assert size > 256 << 20 >= size // copies
    g = torch.Generator(device="cuda").manual_seed(nx)
    rho = 1.0 + 0.02 * (torch.rand((nz, ny, nx), generator=g, device="cuda") - 0.5)
    u = 0.05 * (torch.rand((3, nz, ny, nx), generator=g, device="cuda") - 0.5)
    small.init_equilibrium(rho, u)
    large.init_equilibrium(rho.repeat(copies, 1, 1), u.repeat(1, copies, 1, 1))
    for ctx in (small, large):
        ctx.step(3)
        ctx.macroscopic(macro=True)
    f, rho, u = small.dense_populations(), small.rho, small.u
    assert torch.equal(large.dense_populations(), f.repeat(1, copies, 1, 1))
    assert torch.equal(large.rho, rho.repeat(copies, 1, 1)) and torch.equal(large.u, u.repeat(1, copies, 1, 1))
