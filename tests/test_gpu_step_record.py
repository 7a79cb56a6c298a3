"""pol_step_record: the recorded states and outlet fluxes against the same steps
taken one by one with their full reductions, for windows that start at, inside
and past the run, and more fluxes than its host buffer holds (43 + nz)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pourover_amd import _lib as L
from pourover_amd import workloads as WL
from pourover_amd.engine import HipContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n", [("f32", 32), ("f64", 33), ("f16", 32), ("f32", 70)])
def test_states_and_fluxes(precision, n):
    wl = WL.v60_config(n, precision, perm_field=precision in ("f32", "f64"))
    count = 2 * (43 + n) + 3 if n == 32 and precision == "f32" else 6
    for first in (0, 2, count - 1, count, count + 5):
        print("case: step record %s %d^3 count=%d first=%d" % (precision, n, count, first), flush=True)
        a, b = HipContext(wl.config, wl.geometry.flags), HipContext(wl.config, wl.geometry.flags)
        for ctx in (a, b):
            ctx.init_equilibrium()
            ctx.step(40)
        states = torch.empty((count,) + tuple(a.f_current.shape), dtype=a.f_current.dtype, device=a.device)
        states[0].copy_(a.f_current)
        final = torch.zeros_like(states[0])
        flux = np.full(max(count - first, 1), np.nan)
        st = a.lib.pol_step_record(a.handle, states.data_ptr(), states[0].numel() * states.element_size(), count,
                                   final.data_ptr(), first, flux.ctypes.data if first < count else None,
                                   L.stream_handle())
        L.check(st, a.handle, "pol_step_record")
        torch.cuda.synchronize()
        for i in range(count):
            # (no step writes the slots that hold no cell)
            assert torch.equal(a.dense_populations(states[i]), b.dense_populations()), i
            red = b.step(1, L.POL_WANT_REDUCE)
            if i >= first:  # the same FP64 terms (fewer than 100 outlet cells) in another order
                assert abs(flux[i - first] - red[7]) <= 100 * 2.0 ** -52 * abs(red[7]) + 1e-300, i
                assert red[7] != 0.0
        assert torch.equal(a.dense_populations(final), b.dense_populations())


def test_refused_calls():
    wl = WL.v60_config(32, "f32")
    ctx = HipContext(wl.config, wl.geometry.flags)
    f = ctx.f_current
    out = torch.empty_like(f)
    args = lambda **k: {**dict(states=f.data_ptr(), stride=f.numel() * 4, count=1, final=out.data_ptr(), first=1, flux=None), **k}

    def call(k):
        return ctx.lib.pol_step_record(ctx.handle, k["states"], k["stride"], k["count"], k["final"], k["first"], k["flux"],
                                       L.stream_handle())

    for bad in (dict(states=None), dict(final=None), dict(count=0), dict(first=-1), dict(first=0),
                dict(count=2, stride=0, first=2)):
        assert call(args(**bad)) == L.POL_ERR_INVALID, bad
    assert call(args()) == L.POL_OK
    torch.cuda.synchronize()
