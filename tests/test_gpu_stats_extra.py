"""The field statistics with each combination of a previous density, a
previous velocity and a phase field: the 4-cell form (fields on 16-byte
boundaries) against the one-cell form that a field off that boundary selects."""
from __future__ import annotations

import itertools

import pytest
import torch

from pourover_amd import diagnostics as D
from pourover_amd.engine import HipContext, SolverConfig

pytestmark = pytest.mark.gpu


def _off(t, by):
    """A copy of t that starts `by` elements into its allocation."""
    a = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)
    a[by:].copy_(t.reshape(-1))
    return a[by:].view(t.shape)


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("shape", [(4, 4, 3), (6, 10, 9), (224, 9, 4)])
def test_forms_agree(shape, precision):
    nx, ny, nz = shape
    ctx = HipContext(SolverConfig(nx, ny, nz, precision=precision))
    g = torch.Generator().manual_seed(nx)

    def field(*lead):
        return (torch.rand(lead + (nz, ny, nx), generator=g, dtype=torch.float64) - 0.4).to(ctx.rho)

    ctx.rho.copy_(1.0 + 0.1 * field())
    ctx.u.copy_(0.1 * field(3))
    prev_rho, prev_u, phase = 1.0 + 0.1 * field(), 0.1 * field(3), field()
    for use in itertools.product((False, True), repeat=3):
        if not any(use):
            continue
        given = [t if on else None for t, on in zip((prev_rho, prev_u, phase), use)]
        a, za = D.field_statistics(ctx, *given)
        b, zb = D.field_statistics(ctx, *[None if t is None else _off(t, 1 if precision == "f64" else 3) for t in given])
        sums = {k for k in a if k.startswith(("sum", "mom", "d", "int_water", "int_air", "int_usum", "outlet"))}
        n, eps = nx * ny * nz, 2.0 ** -52
        for k in a:
            # sums of at most n values below 2 in another order; everything else exactly
            assert abs(a[k] - b[k]) <= (2 * n * n * eps if k in sums else 0.0), (use, k, a[k], b[k])
        assert abs(za - zb).max() <= 2 * n * n * eps
        assert (a["drho_prev2"] > 0) == use[0] and (a["du_prev2"] > 0) == use[1] and (a["int_air"] > 0) == (use[2] and nz > 2)
