"""The kernel forms that the size rules take above the last-level cache and that
smaller tests do not reach, on boxes just above their limits: the pressure
drive with the surface tension in the same pass, the drive and the phase step
in FP64 storage, the eddy viscosity in grouped block order.  Bit for bit
against the separate passes, the numpy restatements or the same pass over a
slab of the box that stays in the cache."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import forcing as OF
from oracle import multiphase as OM
from oracle.les_fd import les_fd_viscosity, mask_from_flags
from pourover_amd import _lib as L
from pourover_amd import forcing as FC
from pourover_amd import multiphase as MP
from pourover_amd.engine import HipContext, SolverConfig
from pourover_amd.geometry import link_flags

pytestmark = pytest.mark.gpu

F = np.float32


def _same(a, b, what):
    bits = {4: np.int32, 8: np.int64}[a.itemsize]
    assert a.dtype == b.dtype and a.shape == b.shape and np.array_equal(a.view(bits), b.view(bits)), what


def _box(shape, precision, seed, solid=0.1):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    kind = (rng.random((nz, ny, nx), dtype=F) < solid).astype(np.uint8)
    cfg = SolverConfig(nx, ny, nz, precision=precision, periodic=(False, False, False), force_field=True)
    return rng, kind, HipContext(cfg, link_flags(kind)[0])


def _uniform(rng, lo, hi, shape):
    return (rng.random(shape, dtype=F) * F(hi - lo) + F(lo)).astype(F)


# 44 B a cell in FP32, 72 in FP64: limit at 6.1 / 3.7 million cells
@pytest.mark.parametrize("mode", ["force", "mixed"])
@pytest.mark.parametrize("precision,shape", [("f32", (193, 181, 179)), ("f64", (161, 155, 151))])
def test_drive_with_surface_tension(precision, shape, mode):
    print("case: streaming drive with surface tension %s %s %s" % (precision, shape, mode), flush=True)
    rng, kind, ctx = _box(shape, precision, 21)
    mp = MP.MultiphaseFlow3D(ctx)
    drive = FC.PressureGradientDrive(ctx)
    getattr(drive, "activate_%s_drive" % mode)(True)
    real = np.float64 if precision == "f64" else F
    rho = _uniform(rng, 0.9, 1.1, kind.shape).astype(real)
    rho[12, 10, 11] = real(1e-11)
    bf = _uniform(rng, -1e-3, 1e-3, (3,) + kind.shape).astype(real)
    bf[:, 5, 5, 5] = real(-0.0)
    phi = _uniform(rng, -1.2, 1.2, kind.shape)
    mp._phi[mp._cur].copy_(torch.from_numpy(phi))
    ctx.rho.copy_(torch.from_numpy(rho))

    def body_force():
        ctx.force.copy_(torch.from_numpy(bf))
        drive._pforce.zero_()

    body_force()
    drive.apply(3)
    mp.accumulate_surface_tension_pre_collision()
    pf_two, bf_two = drive._pforce.cpu().numpy(), ctx.force.cpu().numpy()
    body_force()
    mp.accumulate_surface_tension_pre_collision = lambda: pytest.fail("separate passes")
    drive.apply_with_surface_tension(mp, 3)
    _same(drive._pforce.cpu().numpy(), pf_two, "pressure force")
    _same(ctx.force.cpu().numpy(), bf_two, "body force")
    _same(pf_two, OF.pressure_force(rho.astype(F), kind), "pressure force against the restatement")


# FP64: 52 B a cell of the phase step, limit at 5.2 million cells
@pytest.mark.parametrize("shape", [(177, 173, 171), (65, 40, 21)])
def test_phase_step_and_drive_f64(shape):
    """Inputs are FP32 values, so that the FP32 restatements hold: both passes
    compute in FP32 and store the result in the real type."""
    print("case: streaming phase step and pressure drive f64 %s" % (shape,), flush=True)
    rng, kind, ctx = _box(shape, "f64", 22)
    mp = MP.MultiphaseFlow3D(ctx)
    drive = FC.PressureGradientDrive(ctx)
    drive.activate_force_drive(True)
    phi, mu, faces = (_uniform(rng, -1, 1, kind.shape) for _ in range(3))
    rho, u = _uniform(rng, 0.001, 1, kind.shape), _uniform(rng, -0.05, 0.05, (3,) + kind.shape)
    bf = _uniform(rng, -1e-3, 1e-3, u.shape).astype(np.float64)
    for dst, src in ((mp._phi[0], phi), (mp._mu, mu), (mp._phi_new, faces), (ctx.rho, rho), (ctx.u, u), (ctx.force, bf)):
        dst.copy_(torch.from_numpy(src))
    drive.apply_force_drive()
    pf = OF.pressure_force(rho, kind)
    _same(drive._pforce.cpu().numpy(), pf, "pressure force")
    _same(ctx.force.cpu().numpy(), np.where((kind == 0)[None], bf + pf.astype(np.float64), bf), "body force")
    mp.step(1, precollision_applied=True)
    t = lambda a: np.ascontiguousarray(a.transpose(2, 1, 0))
    s = OM.new_state(t(phi), u.transpose(3, 2, 1, 0), t(rho), t(kind), mu=t(mu), phi_new=t(faces))
    OM.update_phase_field(s)
    OM.phase_separation(s)
    s["phi"] = s["phi_new"].copy()
    OM.density_from_phase(s)
    _same(mp._phi[mp._cur].cpu().numpy(), t(s["phi"]), "phi")
    for got, name in ((ctx.rho, "rho"), (mp._phase, "phase")):
        _same(got.cpu().numpy(), t(s[name]).astype(np.float64), name)


# with flags and a phase: FP32 24 B a cell, FP64 44, limits at 11.2 and 6.1 million cells
@pytest.mark.parametrize("precision,shape", [("f32", (227, 225, 223)), ("f64", (187, 181, 183))])
def test_eddy_viscosity(precision, shape):
    print("case: streaming eddy viscosity %s %s" % (precision, shape), flush=True)
    nx, ny, nz = shape
    real = np.float64 if precision == "f64" else F
    rng = np.random.default_rng(23)
    kind = (rng.random((nz, ny, nx), dtype=F) < 0.1).astype(np.uint8)
    u = (rng.standard_normal((3, nz, ny, nx), dtype=F) * F(0.01))
    u[:, nz // 3: nz // 2] *= F(0.01)  # a band below the |S| < 1e-3 cut
    u = u.astype(real)
    phase = _uniform(rng, -1.5, 1.5, kind.shape).astype(real)

    def viscosity(sl):
        """of the planes sl as a box of their own"""
        flags = link_flags(np.ascontiguousarray(kind[sl]))[0]
        n = kind[sl].shape[0]
        ctx = HipContext(SolverConfig(nx, ny, n, precision=precision, periodic=(False, False, False), les=True,
                                      les_fd=True, cs_smag=0.17), flags)
        ctx.u.copy_(torch.from_numpy(np.ascontiguousarray(u[:, sl])))
        ctx.les_phase = torch.from_numpy(np.ascontiguousarray(phase[sl])).cuda()
        ctx._bind_keep_state()
        L.check(ctx.lib.pol_les_viscosity(ctx.handle, None, L.stream_handle()), ctx.handle, "pol_les_viscosity")
        return ctx.nu_sgs.cpu().numpy(), flags, ctx.config

    got, flags, cfg = viscosity(slice(0, nz))
    assert (got > 0).sum() > 1000 and (got[nz // 3 + 1: nz // 2 - 1] > 0).sum() == 0
    if precision == "f32":
        _same(got, les_fd_viscosity(u, mask=mask_from_flags(flags), phase=phase, cs=cfg.cs_smag, nu_max=cfg.nu_sgs_max),
              "restatement")
    for z0 in (0, nz // 2 - 7, nz - 21):
        part = viscosity(slice(z0, z0 + 21))[0]
        _same(got[z0 + 1: z0 + 20], part[1:20], "planes %d on" % z0)
