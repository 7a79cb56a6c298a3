"""The population scan of pol_field_stats (k_pop_nonfinite): NaN and infinite
populations of the non-solid cells, counted exactly, for each storage, on the
compact and the dense layout, from none to every value of the state."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd import _lib as L
from pourover_amd import diagnostics as D
from pourover_amd import workloads as WL
from pourover_amd.engine import HipContext, SolverConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [0.0, 1e-5, 0.3, 1.0])
@pytest.mark.parametrize("precision,compact", [("f32", True), ("f32", False), ("f16", True), ("bf16", True), ("f64", True)])
def test_counts_of_planted_values(precision, compact, share):
    print("case: population scan 33^3 %s compact=%s share=%g" % (precision, compact, share), flush=True)
    wl = WL.v60_config(33, precision)
    ctx = HipContext(wl.config, wl.geometry.flags, compact=compact)
    ctx.init_equilibrium()
    ctx.step(3, L.POL_WANT_MACRO)
    rng = np.random.default_rng(7)
    pick = torch.from_numpy(rng.random(tuple(ctx.f_current.shape))).to(ctx.device)
    f = ctx.f_current
    f[pick < share] = float("nan")
    f[pick < share / 2] = float("inf")
    f[pick < share / 4] = float("-inf")
    open_cell = torch.from_numpy(wl.geometry.kind != L.POL_KIND_SOLID).to(ctx.device)
    seen = ctx.dense_populations()[:, open_cell]
    for _ in range(2):  # a second call counts afresh
        s, _ = D.field_statistics(ctx, populations=True)
        assert s["fluid_pop_nan"] == int(torch.isnan(seen).sum()) and s["fluid_pop_inf"] == int(torch.isinf(seen).sum())
    if share >= 0.3:  # (1e-5 of 167 808 values may fall on solid cells only)
        assert s["fluid_pop_nan"] > 0 and s["fluid_pop_inf"] > 0


@pytest.mark.parametrize("shape", [(2, 2, 2), (17, 5, 3)])
def test_counts_without_flags(shape):
    ctx = HipContext(SolverConfig(*shape))
    ctx.init_equilibrium()
    ctx.f_current[3, -1] = float("nan")
    ctx.f_current[18, -1] = float("-inf")
    s, _ = D.field_statistics(ctx, populations=True)
    assert s["fluid_pop_nan"] == 1 and s["fluid_pop_inf"] == 1


def test_calls_with_and_without_the_scan():
    """The scan's counts belong to the call that asks for them, and the other
    statistics and the plane profile do not depend on it."""
    wl = WL.v60_config(33, "f32")
    ctx = HipContext(wl.config, wl.geometry.flags)
    ctx.init_equilibrium()
    ctx.step(3, L.POL_WANT_MACRO)
    clean = ctx.f_current.clone()
    at = int(ctx.layout.run_slots[len(ctx.layout.run_slots) // 2])
    while wl.geometry.kind.reshape(-1)[ctx.layout.slot_dense[at]] == L.POL_KIND_SOLID:
        at += 1
    want, profile = D.field_statistics(ctx)
    for planted in (3, 0, 5):
        ctx.f_current.copy_(clean)
        ctx.f_current.view(19, -1)[:planted, at] = float("nan")
        s, z = D.field_statistics(ctx, populations=True)
        assert s["fluid_pop_nan"] == planted and s["fluid_pop_inf"] == 0
        plain, z2 = D.field_statistics(ctx)
        assert plain["fluid_pop_nan"] == 0 and plain["fluid_pop_inf"] == 0
        for key in want:
            if not key.startswith("fluid_pop"):
                assert s[key] == plain[key] == want[key], key
        if profile is not None:
            assert np.array_equal(z, profile) and np.array_equal(z2, profile)
