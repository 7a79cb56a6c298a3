"""The phase step and the pressure drive above the last-level cache (stores past
the cache) against the numpy restatements, bit for bit, on a box whose extents
are no multiples of a wave."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import forcing as OF
from oracle import multiphase as OM
from pourover_amd import forcing as FC
from pourover_amd import multiphase as MP
from pourover_amd.engine import HipContext, SolverConfig
from pourover_amd.geometry import link_flags

pytestmark = pytest.mark.gpu

F = np.float32


def _same(a, b):
    assert a.shape == b.shape and np.array_equal(a.view(np.int32), b.view(np.int32))


@pytest.mark.parametrize("shape", [(203, 205, 211), (65, 40, 21)])  # 8.8 M cells (281 MB per pass); cached
def test_one_step(shape):
    nx, ny, nz = shape
    print("case: streaming phase step and pressure drive %s" % (shape,), flush=True)
    rng = np.random.default_rng(nx)
    kind = (rng.random((nz, ny, nx)) < 0.1).astype(np.uint8)  # scattered solid cells
    cfg = SolverConfig(nx, ny, nz, periodic=(False, False, False), force_field=True)
    ctx = HipContext(cfg, link_flags(kind)[0])
    mp = MP.MultiphaseFlow3D(ctx)
    drive = FC.PressureGradientDrive(ctx)
    drive.activate_force_drive(True)
    phi = rng.uniform(-1, 1, (nz, ny, nx)).astype(F)
    mu, faces = rng.uniform(-1, 1, phi.shape).astype(F), rng.uniform(-1, 1, phi.shape).astype(F)
    rho, u = rng.uniform(0.001, 1, phi.shape).astype(F), rng.uniform(-0.05, 0.05, (3,) + phi.shape).astype(F)
    bf = rng.uniform(-1e-3, 1e-3, u.shape).astype(F)
    for dst, src in ((mp._phi[0], phi), (mp._mu, mu), (mp._phi_new, faces), (ctx.rho, rho), (ctx.u, u), (ctx.force, bf)):
        dst.copy_(torch.from_numpy(src))
    drive.apply_force_drive()
    _same(drive._pforce.cpu().numpy(), OF.pressure_force(rho, kind))
    _same(ctx.force.cpu().numpy(), OF.accumulate(bf, OF.pressure_force(rho, kind), kind))
    mp.step(1, precollision_applied=True)
    t = lambda a: np.ascontiguousarray(a.transpose(2, 1, 0))
    s = OM.new_state(t(phi), u.transpose(3, 2, 1, 0), t(rho), t(kind), mu=t(mu), phi_new=t(faces))
    OM.update_phase_field(s)
    OM.phase_separation(s)
    s["phi"] = s["phi_new"].copy()
    OM.density_from_phase(s)
    _same(mp._phi[mp._cur].cpu().numpy(), np.ascontiguousarray(s["phi"].transpose(2, 1, 0)))
    _same(ctx.rho.cpu().numpy(), np.ascontiguousarray(s["rho"].transpose(2, 1, 0)))
    _same(mp._phase.cpu().numpy(), np.ascontiguousarray(s["phase"].transpose(2, 1, 0)))
