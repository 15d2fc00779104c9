"""State transfers and point batches at the sizes where their route changes
(pinned buffer up to 256 KB, one copy, ranges of leaves on 4 and 8 streams):
a state comes back as written (FP64) or rounded once (FP32), whatever the
leaf count; a large batch of fluxes equals its parts, and calls from several
threads on one context equal calls in turn; device memory reused by a new mesh
or a smaller one carries nothing over."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import charm_3d_amd as CA

pytestmark = pytest.mark.gpu


def mesh_of(n_target, level):
    """a uniform level with as many leaves refined as n_target needs"""
    f = CA.Forest.uniform(level)
    k = max(0, (n_target - f.n + 6) // 7)
    flags = np.zeros(f.n, np.int8)
    flags[:k] = 1
    if k:
        f.adapt(flags, level + 1)
    return f


# leaves: below and above 256 KB (1,638 of 20 words), 12 MB (78,643) and 64 MB (419,430)
SIZES = [(1, 1), (3, 512), (3, 1600), (3, 1700), (5, 70000), (5, 80000), (6, 400000), (6, 430000)]


@pytest.mark.parametrize("precision", [CA.FP64, CA.FP32])
@pytest.mark.parametrize("level,n", SIZES)
def test_state_round_trip(level, n, precision):
    f = mesh_of(n, level)
    cfg = CA.make_config(flux="HLLC", precision=precision)
    print(f"[transfers] leaves={f.n} precision={precision}", flush=True)
    ctx = CA.GpuContext(cfg)
    ctx.upload_mesh(f.flatten(*CA.recommended_chunks(cfg)))
    rng = np.random.default_rng(n)
    for _ in range(2):
        u = rng.normal(size=(f.n, 5, 4))
        ctx.set_state(u)
        want = u if precision == CA.FP64 else u.astype(np.float32).astype(np.float64)
        np.testing.assert_array_equal(ctx.get_state(), want)


def test_contexts_share_the_transfer_streams():
    """several threads, a context each, and contexts that come and go"""
    f = mesh_of(80000, 5)
    cfg = CA.make_config(flux="HLLC", precision=CA.FP64)
    mesh = f.flatten(*CA.recommended_chunks(cfg))

    def run(seed):
        u = np.random.default_rng(seed).normal(size=(f.n, 5, 4))
        for _ in range(2):
            ctx = CA.GpuContext(cfg)
            ctx.upload_mesh(mesh)
            for _ in range(3):
                ctx.set_state(u)
                if not np.array_equal(ctx.get_state(), u):
                    return False
            ctx.close()
        return True

    with ThreadPoolExecutor(3) as ex:
        assert all(ex.map(run, range(3)))
    assert run(9)


def points(n, seed):
    rng = np.random.default_rng(seed)
    r, p = rng.uniform(0.5, 2, n), rng.uniform(0.5, 2, n)
    v = rng.normal(size=(3, n))
    nn = rng.normal(size=(n, 3))
    return np.stack([r, *v, p, np.ones(n)], 1), nn / np.linalg.norm(nn, axis=1, keepdims=True)


@pytest.mark.parametrize("flux", ["HLLC", "GODUNOV"])
def test_flux_batches_of_every_route_agree(flux):
    ctx = CA.GpuContext(CA.make_config(flux=flux, precision=CA.FP64))
    n = 4000                                    # 640 KB: device buffers
    (pl, nn), (pr, _) = points(n, 1), points(n, 2)
    whole = ctx.flux_batch(flux, pl, pr, nn)
    assert np.isfinite(whole).all()
    cuts = [0, 1, 64, 65, 700, 2300, n]         # 1,638 points are 256 KB
    parts = list(zip(cuts, cuts[1:]))
    for a, b in parts:
        np.testing.assert_array_equal(ctx.flux_batch(flux, pl[a:b], pr[a:b], nn[a:b]), whole[a:b])
    with ThreadPoolExecutor(4) as ex:
        got = list(ex.map(lambda s: ctx.flux_batch(flux, pl[s[0]:s[1]], pr[s[0]:s[1]], nn[s[0]:s[1]]), parts * 5))
    for (a, b), q in zip(parts * 5, got):
        np.testing.assert_array_equal(q, whole[a:b])


def test_reused_device_memory_carries_nothing_over():
    cfg = CA.make_config(flux="HLLC", limiter=True, precision=CA.FP64)

    def run(ctx, level):
        f = CA.Forest.uniform(level)
        u = np.zeros((f.n, 5, 4))
        rng = np.random.default_rng(level)
        u[:, 4, 0] = 1 + 0.1 * rng.uniform(size=f.n)
        u[:, 3, 0] = 2.5 + 0.1 * rng.uniform(size=f.n)
        ctx.upload_mesh(f.flatten(*CA.recommended_chunks(cfg)))
        np.testing.assert_array_equal(ctx.get_state(), 0.0)     # a new mesh starts from zeros
        ctx.set_state(u)
        ctx.step("NS", 1e-4, 3)
        return ctx.get_state()

    kept = CA.GpuContext(cfg)
    for level in (4, 3, 4, 2, 3):
        np.testing.assert_array_equal(run(kept, level), run(CA.GpuContext(cfg), level))
