"""The stage VJP at the sizes where its kernels change (by leaves up to 12,000
leaves in FP32, 24,000 with two species, by chunks beyond; by leaves in FP64,
but for HLLC with two species with two workgroups per CU beyond 24,000, LF and
CD with one species beyond 6,000, and a thread per leaf beyond 65,536 without
hanging faces): <S_u^T x, v> in FP64 against the
central difference of <x, S(u)> to 1e-7, one leaf to 32,768, hanging faces, a
leaf that is its own periodic neighbour; FP32 against FP64 to 1e-5."""
import numpy as np
import pytest

import charm_3d_amd as CA
from test_gpu_parity import device
from test_gpu_small_mesh import BND, PAR, shell, state

pytestmark = pytest.mark.gpu


def setup(mesh, flux, nc, precision, periodic=False):
    leaves = shell(*mesh)
    kw = dict(model="NS", limiter=False, flux=flux, precision=precision, grav=(0.1, -0.2, 0.3), bnd=BND, bnd_param=PAR)
    if periodic:
        kw.update(bnd=("PERIODIC",) * 6, bnd_param=[None] * 6)
    if nc == 2:
        kw.update(eos="MIX", comp_m=(CA.GAS_R, 0.5 * CA.GAS_R), comp_cp=(3.5, 5.0))
        if not periodic:
            kw["bnd_param"] = [(0.4, 0.1, 0.0, 1.1, 1.0, 0.7, 0.3), None, None, None, (0.9,), None]
    cfg = CA.make_config(**kw)
    u = state(len(leaves), nc)
    print(f"[adj_leaves] {mesh} {flux} nc={nc} precision={precision} leaves={len(leaves)}", flush=True)
    ctx = device(cfg, leaves, (periodic,) * 3, u)
    return ctx, u, 0.05 * 2.0 ** -(mesh[0] + mesh[1])


# one leaf to 32,768; with hanging faces near 200, 3,872, 9,192 and 19,104 leaves
MESHES = [(0, 0), (1, 0), (2, 0), (2, 1), (3, 1), (3, 2), (4, 1), (5, 0)]


@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("flux,nc", [("LF", 1), ("HLLC", 1), ("CD", 2), ("HLLC", 2)])
def test_stage_vjp_against_differences(mesh, flux, nc):
    for periodic in (False, True):
        if periodic and mesh[1]:
            continue
        ctx, u, dt = setup(mesh, flux, nc, CA.FP64, periodic)
        rng = np.random.default_rng(3)
        x = rng.normal(size=u.shape)
        v = rng.normal(size=u.shape) * np.abs(u).max(axis=0, keepdims=True)
        g = ctx.stage_vjp(dt, u, x)
        # rounding leaves 1e-16 / h = 1e-8 of the root mean square of the terms.  A
        # larger h meets the kinks of |u_n| and of max(|u| + c): a point lies within
        # h of one with a chance of about h / 0.1, so that at h = 1e-6 one of the
        # 70,000 points of 3,872 leaves does, an error of one term in sqrt(70,000)
        # (1.3e-5 seen); at 1e-8 none is expected up to 32,768 leaves
        h, s = 1e-8, []
        for sg in (1, -1):
            ctx.set_state(u + sg * h * v)
            ctx.step("EULER", dt, 1)
            s.append(ctx.get_state())
        fd = (x * (s[0] - s[1])).sum() / (2 * h)
        # a random x and v may cancel in the sum
        scale = max(abs(fd), np.sqrt(((g * v) ** 2).sum()))
        assert abs((g * v).sum() - fd) <= 1e-7 * scale, ((g * v).sum(), fd, scale)
        np.testing.assert_array_equal(ctx.stage_vjp(dt, u, x), g)
        ctx.close()


@pytest.mark.parametrize("mesh", [(3, 1), (3, 2), (4, 1), (5, 0), (5, 1), (6, 0)])
@pytest.mark.parametrize("flux,nc", [("LF", 1), ("HLLC", 2)])
def test_fp32_stage_vjp_close_to_fp64(mesh, flux, nc):
    out = []
    for prec in (CA.FP64, CA.FP32):
        ctx, u, dt = setup(mesh, flux, nc, prec)
        x = np.random.default_rng(5).normal(size=u.shape)
        out.append(ctx.stage_vjp(dt, u, x))
        ctx.close()
    d = np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0])
    assert d < 1e-5, d
