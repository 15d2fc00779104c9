"""Meshes large enough for the kernels that the small ones of the other tests
do not reach: the chunk stage kernel with viscous terms (beyond 12,000 leaves)
and with the exact Riemann solver (beyond 24,000), against the oracle and FP32
against FP64; the checkpointed adjoint by chunks (FP32, beyond 24,000 leaves)
and with a thread per leaf (FP64, beyond 65,536 without hanging faces), with
the inlet's parameters."""
import numpy as np
import pytest

import charm_3d_amd as CA
import charm_3d_amd.workloads as W
import oracle_lib as OL
import test_gpu_ns as NS
from test_gpu_parity import device, oracle_cfg
from test_gpu_small_mesh import BND, PAR, shell, state

pytestmark = pytest.mark.gpu

SI = [[20.0, 5.0, 0.0, 320.0, 1.0e5], None, [310.0], None, [290.0], None]
ND = [[0.3, 0.1, 0.0, 1.1, 1.0], None, [1.05], None, [0.95], None]


def viscous_case(name, leaves, prec):
    """configuration, state, and the size of p, of the viscosity and of the
    conductivity times T"""
    rng = np.random.default_rng(9)
    if name == "poly":
        cfg = NS.cfg_poly(prec, bnd=NS.WALLS, params=ND)
        return cfg, NS.state(leaves, rng, cfg, 1.0, 1.0, (0.3, 0.2, 0.1)), 1.0, 0.05, 0.1
    if name == "mix":
        cfg = NS.cfg_mix(prec, bnd=NS.WALLS, params=SI)
        return cfg, NS.state(leaves, rng, cfg, 300.0, 1.0e5, (20.0, 10.0, 5.0)), 1.0e5, 1.8e-5, 7.0
    cfg = W.c4_config(prec)
    return cfg, W.project_p1(leaves, W.c4_state_fn(cfg), 8), 101325.0, 5e-5, 100.0


@pytest.mark.parametrize("name", ["poly", "mix", "hot spot"])
def test_viscous_residual(name):
    leaves = shell(4, 1)
    assert len(leaves) > 12000
    out = {}
    for prec in (CA.FP64, CA.FP32):
        cfg, u, p, mu, kt = viscous_case(name, leaves, prec)
        print(f"[sizes] {name} n={len(leaves)} precision={prec}", flush=True)
        ctx = device(cfg, leaves, (False,) * 3, u)
        out[prec] = ctx.residual()
        ctx.close()
        if prec == CA.FP64:
            sim = OL.OracleSim(oracle_cfg(cfg), leaves)
            sim.set_state(u)
            assert NS.var_err(out[prec], sim.ns_residual()) <= 1e-11
    # FP32 rounding, in units of 2^-24 of a face's flux: the momentum flux p + rho
    # u^2; for energy and mass the traces' rounding enters with the wave speeds,
    # c (E + p) and c rho; the viscous fluxes are differences of two traces over
    # h, 2 mu |u| / h and 2 (mu u^2 + k T) / h.  A point's flux takes some ten
    # roundings of up to half a unit, 2 in the mean, a leaf's integrals six faces
    # and the volume term
    rho, h = u[:, 4:, 0].sum(1), 2.0 ** -leaves[:, 3].astype(float)
    c, u2 = np.sqrt(1.4 * p / rho), (u[:, :3, 0] ** 2).sum(1) / rho ** 2
    f = np.stack([p + rho * u2 + 2 * mu * np.sqrt(u2) / h] * 3 + [c * (u[:, 3, 0] + p) + 2 * (mu * u2 + kt) / h] +
                 [c * rho] * (u.shape[1] - 4), 1)
    err = np.abs(out[CA.FP32] - out[CA.FP64]) / (h[:, None, None] ** 2 * f[:, :, None]) * 2.0 ** 24
    rms = np.sqrt((err ** 2).mean(axis=(0, 2)))
    print(f"[sizes] {name} FP32 units {np.round(rms, 2)}", flush=True)
    assert rms.max() <= 2.0 * np.sqrt(7.0), rms


@pytest.mark.parametrize("mesh,nc", [((5, 0), 1), ((5, 0), 2), ((4, 2), 2), ((5, 0), 3)])
def test_exact_solver_residual(mesh, nc):
    leaves = shell(*mesh)
    assert len(leaves) > 24000
    kw = dict(flux="GODUNOV", bnd=BND, bnd_param=PAR, grav=(0.1, -0.2, 0.3))
    if nc > 1:
        kw.update(eos="MIX", comp_m=tuple(CA.GAS_R * m for m in (1.0, 0.5, 0.8)[:nc]), comp_cp=(3.5, 5.0, 4.0)[:nc])
        kw["bnd_param"] = [(0.4, 0.1, 0.0, 1.1, 1.0) + ((0.7, 0.3), (0.5, 0.3, 0.2))[nc - 2]] + PAR[1:]
    u = state(len(leaves), nc)
    out = {}
    for prec in (CA.FP64, CA.FP32):
        print(f"[sizes] exact solver n={len(leaves)} nc={nc} precision={prec}", flush=True)
        cfg = CA.make_config(precision=prec, **kw)
        ctx = device(cfg, leaves, (False,) * 3, u)
        out[prec] = ctx.residual()
        ctx.close()
        if prec == CA.FP64:
            sim = OL.OracleSim(oracle_cfg(cfg), leaves)
            sim.set_state(u)
            assert NS.var_err(out[prec], sim.residual()) <= 1e-9
    # FP32 rounding of O(1) fluxes over a leaf's six faces and eight points
    assert np.linalg.norm(out[CA.FP32] - out[CA.FP64]) <= 2e-5 * np.linalg.norm(out[CA.FP64])


LO, HI = (0.0, 0.0, 0.0), (0.45, 1.0, 1.0)
STEPS = 4


def pulse(level, precision, inlet=(0.5, 1.0, 1.0)):
    cfg, lv, u0, per = W.c5_pulse(level, precision, inlet)
    print(f"[sizes] adjoint level {level} precision={precision}", flush=True)
    return device(cfg, lv, per, u0), 0.08 * 2.0 ** -level


def test_chunk_adjoint_close_to_fp64():
    """FP32 by chunks, every state kept and checkpoints every 3 steps: the same
    bits, within the small meshes' 1e-4 of the FP64 adjoint by leaves"""
    ctx, dt = pulse(5, CA.FP64)
    ref = ctx.adjoint(dt, STEPS, LO, HI, ckpt=3, theta_face=0)
    ctx.close()
    ctx, dt = pulse(5, CA.FP32)
    assert ctx.n > 24000
    kept = ctx.adjoint(dt, STEPS, LO, HI, ckpt=0, theta_face=0)
    ctx.close()
    ctx, dt = pulse(5, CA.FP32)
    got = ctx.adjoint(dt, STEPS, LO, HI, ckpt=3, theta_face=0)
    ctx.close()
    assert got[0] == kept[0] and np.array_equal(got[1], kept[1]) and np.array_equal(got[2], kept[2])
    assert abs(got[0] - ref[0]) <= 1e-5 * abs(ref[0])
    assert np.linalg.norm(got[1] - ref[1]) <= 1e-4 * np.linalg.norm(ref[1])
    np.testing.assert_allclose(got[2], ref[2], rtol=1e-4)


def test_thread_per_leaf_adjoint_against_differences():
    """FP64 at level 6: the inlet's gradient and the initial state's along one
    direction against central differences, as on the small meshes"""
    inlet = np.array([0.5, 1.0, 1.0])
    ctx, dt = pulse(6, CA.FP64)
    u0 = ctx.get_state()
    assert ctx.n > 65536
    kept = ctx.adjoint(dt, STEPS, LO, HI, ckpt=0, theta_face=0)
    ctx.set_state(u0)
    J, g, th, _, _ = ctx.adjoint(dt, STEPS, LO, HI, ckpt=3, theta_face=0)
    assert J == kept[0] and np.array_equal(g, kept[1]) and np.array_equal(th, kept[2])
    v = np.random.default_rng(5).normal(size=u0.shape) * np.abs(u0).max(axis=0, keepdims=True)
    s = []
    for sg in (1, -1):
        ctx.set_state(u0 + sg * 1e-7 * v)
        s.append(ctx.objective(dt, STEPS, LO, HI))
    ctx.close()
    fd, ad = (s[0] - s[1]) / 2e-7, float((g * v).sum())
    print(f"[sizes] state {ad:.12e} {fd:.12e}", flush=True)
    assert abs(ad - fd) <= 1e-5 * max(abs(fd), np.sqrt(((g * v) ** 2).sum()))
    for k in range(3):
        h, s = 1e-6 * max(abs(inlet[k]), 1.0), []
        for sg in (1, -1):
            p = inlet.copy()
            p[k] += sg * h
            ctx, _ = pulse(6, CA.FP64, tuple(p))
            s.append(ctx.objective(dt, STEPS, LO, HI))
            ctx.close()
        fd = (s[0] - s[1]) / (2 * h)
        print(f"[sizes] theta {k} {th[k]:.12e} {fd:.12e}", flush=True)
        assert abs(th[k] - fd) <= 1e-5 * abs(fd), k
