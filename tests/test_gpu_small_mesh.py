"""Small meshes, whose chunks a context cuts into pieces and whose smallest
run one thread per quadrature point: FP64 residuals against the oracle to
1e-12 at the sizes where the rule changes, uniform and with hanging faces,
every flux, one and two species, viscous with polynomial cp; FP32 against
FP64 (bound in the test); the caller's chunk sizes change nothing."""
import numpy as np
import pytest

import charm_3d_amd as CA
import oracle_lib as OL
from test_gpu_ns import cfg_mix, cfg_poly, var_err
from test_gpu_parity import oracle_cfg

pytestmark = pytest.mark.gpu

BND = ("INLET", "OUTLET", "WALL_SLIP", "OUTLET", "WALL_NO_SLIP", "OUTLET")
PAR = [(0.4, 0.1, 0.0, 1.1, 1.0), None, None, None, (0.9,), None]


def shell(level, depth):
    """a uniform level refined `depth` times about a sphere, 2:1 balanced"""
    f = CA.Forest.uniform(level)
    for d in range(depth):
        lv = f.leaves().astype(np.float64)
        h = 2.0 ** -lv[:, 3]
        r = np.sqrt(((lv[:, :3] / CA.ROOT_LEN + 0.5 * h[:, None] - 0.5) ** 2).sum(1))
        f.adapt(((np.abs(r - 0.3) < (3.0 - 1.8 * d) * h) & (lv[:, 3] == level + d)).astype(np.int8), level + depth)
    return f.leaves()


def state(n, nc, seed=5):
    rng = np.random.default_rng(seed)
    u = np.zeros((n, 4 + nc, 4))
    y = rng.uniform(0.2, 0.8, (n, nc))
    rho = 1 + 0.1 * rng.uniform(-1, 1, n)
    u[:, 4:, 0] = rho[:, None] * y / y.sum(1, keepdims=True)
    vel = 0.3 * rng.normal(size=(n, 3))
    u[:, :3, 0] = rho[:, None] * vel
    u[:, 3, 0] = 2.5 * (1 + 0.1 * rng.uniform(-1, 1, n)) + 0.5 * rho * (vel ** 2).sum(1)
    u[:, :, 1:] = 0.05 * rng.normal(size=(n, 4 + nc, 3)) * np.abs(u[:, :, :1])
    return u


def residual(cfg, leaves, u, chunks=None):
    ctx = CA.GpuContext(cfg)
    ctx.upload_mesh(CA.Forest.from_leaves(leaves).flatten(*(chunks or CA.recommended_chunks(cfg))))
    ctx.set_state(u)
    return ctx.residual()


# uniform; with hanging faces: 3,872, 9,192 and 19,104 leaves or near them
MESHES = [(1, 0), (3, 0), (4, 0), (3, 1), (3, 2), (4, 1)]


@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("flux,nc", [("LF", 1), ("HLLC", 1), ("CD", 2), ("GODUNOV", 2)])
def test_small_mesh_residual(mesh, flux, nc):
    kw = dict(flux=flux, bnd=BND, bnd_param=PAR, grav=(0.1, -0.2, 0.3))
    if nc == 2:
        kw.update(eos="MIX", comp_m=(CA.GAS_R, 0.5 * CA.GAS_R), comp_cp=(3.5, 5.0))
    leaves = shell(*mesh)
    u = state(len(leaves), nc)
    print(f"[gpu] n={len(leaves)} {flux} nc={nc}", flush=True)
    cfg = CA.make_config(precision=CA.FP64, **kw)
    got = residual(cfg, leaves, u)
    sim = OL.OracleSim(oracle_cfg(cfg), leaves)
    sim.set_state(u)
    assert var_err(got, sim.residual()) <= (1e-9 if flux == "GODUNOV" else 1e-12)
    assert var_err(residual(cfg, leaves, u, (1, 24)), got) <= 1e-13
    # FP32 rounding of O(1) fluxes over a leaf's six faces and eight points
    got32 = residual(CA.make_config(precision=CA.FP32, **kw), leaves, u)
    assert np.linalg.norm(got32 - got) <= 2e-5 * np.linalg.norm(got)


@pytest.mark.parametrize("mesh", [(2, 1), (3, 2)])
@pytest.mark.parametrize("make", [cfg_poly, cfg_mix])
def test_small_mesh_viscous_residual(mesh, make):
    leaves = shell(*mesh)
    cfg = make()
    rng = np.random.default_rng(9)
    nc = cfg.n_comp
    n = len(leaves)
    if nc == 1:
        u = state(n, 1)
    else:
        # near 400 K, 1 atm: e of about 3e5 J/kg
        y = rng.uniform(0.3, 0.7, n)
        rho = 0.9 * (1 + 0.02 * rng.uniform(-1, 1, n))
        u = np.zeros((n, 6, 4))
        u[:, 3, 0] = rho * 3.0e5 * (1 + 0.02 * rng.uniform(-1, 1, n))
        u[:, 4, 0], u[:, 5, 0] = rho * y, rho * (1 - y)
        u[:, :3, 0] = rho[:, None] * 10.0 * rng.normal(size=(n, 3))
        u[:, :, 1:] = 0.01 * rng.normal(size=(n, 6, 3)) * np.abs(u[:, :, :1])
    print(f"[gpu] n={n} viscous nc={nc}", flush=True)
    got = residual(cfg, leaves, u)
    sim = OL.OracleSim(oracle_cfg(cfg), leaves)
    sim.set_state(u)
    assert var_err(got, sim.ns_residual()) <= 1e-11


def test_branch_flips_between_fluxes():
    """contexts whose fluxes cut one mesh into other pieces: every interior
    (sub)face once, from either context"""
    leaves = shell(4, 1)
    assert 12000 < len(leaves) <= 24000
    print(f"[gpu] n={len(leaves)} branch flips", flush=True)
    mesh = CA.Forest.from_leaves(leaves).flatten(85, 256)
    u = state(len(leaves), 2)
    ctx = []
    for flux in ("GODUNOV", "LF"):
        ctx.append(CA.GpuContext(CA.make_config(precision=CA.FP64, flux=flux, eos="MIX",
                                                comp_m=(CA.GAS_R, 0.5 * CA.GAS_R), comp_cp=(3.5, 5.0))))
        ctx[-1].upload_mesh(mesh)
        ctx[-1].set_state(u)
    interior = int((mesh.faces()[:, 1] >= 0).sum())
    for a, b in (ctx, ctx[::-1]):
        assert a.hllc_branch_flips(b) == (6 * interior, 0)
