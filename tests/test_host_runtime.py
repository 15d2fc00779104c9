"""The host side of the GPU entry points on the CPU, over a stand-in for the
HIP calls (host_hip.c, loaded ahead of the library in a process of its own):
what they refuse, what they leave queued, allocated and changed."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def hip():
    h = C.CDLL(os.environ["HOST_HIP"], mode=C.RTLD_GLOBAL)
    h.hh_limit.argtypes, h.hh_live.restype = [C.c_size_t], C.c_size_t
    return h


def context(level, precision=0, flux="HLLC", chunks=(128, 512), mesh=None, **kw):
    import charm_3d_amd as CA
    ctx = CA.GpuContext(CA.make_config(precision=precision, flux=flux, **kw))
    ctx.upload_mesh(mesh or CA.Forest.uniform(level).flatten(*chunks))
    return ctx


def null_arrays():
    """a null state is an argument error at every size of transfer"""
    import charm_3d_amd as CA
    L = CA.lib()
    for level in (1, 4, 6):              # pinned, one copy, ranges
        ctx = context(level)
        for fn in (L.charm_gpu_set_state, L.charm_gpu_get_state, L.charm_gpu_residual):
            assert fn(ctx.h, None, ctx.n) == -1, fn.__name__
            assert b"null" in L.charm_gpu_last_error()
        ctx.close()


def branch_flips_across_fluxes():
    """two contexts on one mesh of some 13,700 leaves, which the exact solver's
    and the other fluxes' contexts of two species cut into other pieces; other
    leaves, and the same leaves flattened otherwise, are refused"""
    import charm_3d_amd as CA
    lv = CA.Forest.uniform(4)
    lv.adapt((np.arange(lv.n) % 3 == 0).astype(np.int8), 5)
    assert 12000 < lv.n < 24000, lv.n
    mesh = lv.flatten(85, 256)
    kw = dict(eos="MIX", comp_m=(CA.GAS_R, 0.5 * CA.GAS_R), comp_cp=(3.5, 5.0))
    a, b = (context(0, flux=f, mesh=mesh, **kw) for f in ("GODUNOV", "HLLC"))
    assert a.hllc_branch_flips(b) == (0, 0) and b.hllc_branch_flips(a) == (0, 0)
    for other in (context(4, chunks=(85, 256), **kw), context(0, mesh=lv.flatten(100, 300), **kw)):
        with pytest.raises(CA.CharmError, match="same mesh"):
            a.hllc_branch_flips(other)


def failed_uploads():
    """an upload that runs out of device memory at any of its allocations
    leaves no work queued on the blocks it gives back, and no mesh"""
    import charm_3d_amd as CA
    mesh = CA.Forest.uniform(3).flatten(128, 512)
    ctx = context(3)
    used = HIP.hh_live()
    ctx.close()
    failed = 0
    for limit in range(used // 40, used, used // 40):
        ctx = CA.GpuContext(CA.make_config(precision=CA.FP64))
        HIP.hh_limit(limit)
        try:
            ctx.upload_mesh(mesh)
        except CA.CharmError as e:
            failed += 1
            assert "hipMalloc" in str(e) and HIP.hh_queued() == 0, HIP.hh_queued()
            with pytest.raises(CA.CharmError, match="no mesh"):
                ctx.run(0.1, 1)
        HIP.hh_limit(1 << 32)
        ctx.upload_mesh(mesh)
        ctx.run(0.1, 1)
        ctx.close()
    assert failed > 30 and HIP.hh_live() == 0


def refused_remesh():
    """a mesh that remesh refuses leaves the context its mesh and state"""
    import charm_3d_amd as CA
    ctx = context(3)
    n = ctx.n
    with pytest.raises(CA.CharmError, match="LDS"):
        ctx.remesh(CA.Forest.uniform(3).flatten(170, 1000), np.arange(n))
    assert ctx.n == n
    ctx.adjoint(0.1, 1, [0.0] * 3, [1.0] * 3, ckpt=0)    # copies the state


def blocks_kept_by_other_contexts():
    """an allocation that would fail is served from what other contexts keep
    of freed blocks, and a context that is gone is not asked"""
    import charm_3d_amd as CA
    gone, a, b = context(4), context(5), context(1)
    gone.close()
    a.upload_mesh(CA.Forest.uniform(1).flatten())        # level 5's blocks are free now
    HIP.hh_limit(HIP.hh_live() + 65536)
    b.upload_mesh(CA.Forest.uniform(5).flatten(128, 512))
    with pytest.raises(CA.CharmError, match="out of memory"):
        a.upload_mesh(CA.Forest.uniform(5).flatten(128, 512))
    HIP.hh_limit(1 << 32)
    a.close()
    b.close()
    assert HIP.hh_live() == 0


def transfer_streams():
    """streams for large transfers are kept across contexts, are shared, and go
    back when memory runs out"""
    import charm_3d_amd as CA
    mesh = CA.Forest.uniform(6).flatten(170, 512)        # a state of 42 MB
    u = np.zeros((262144, 5, 4))
    for _ in range(3):
        ctx = context(0, mesh=mesh)
        ctx.set_state(u)
        ctx.close()
        assert HIP.hh_streams() == 4
    a, b = context(0, mesh=mesh), context(0, mesh=mesh)
    a.set_state(u)
    b.set_state(u)
    assert HIP.hh_streams() == 4 + 2
    HIP.hh_limit(HIP.hh_live())
    with pytest.raises(CA.CharmError, match="out of memory"):
        a.objective(0.1, 1000, [0.0] * 3, [1.0] * 3)
    assert HIP.hh_streams() == 2
    HIP.hh_limit(1 << 32)
    np.testing.assert_array_equal(a.get_state(), u)
    assert HIP.hh_streams() == 4 + 2


CASES = {f.__name__: f for f in (null_arrays, branch_flips_across_fluxes, failed_uploads, refused_remesh,
                                 blocks_kept_by_other_contexts, transfer_streams)}


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "host_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-pthread", "-o", so,
                    os.path.join(HERE, "host_hip.c")], check=True)
    return so


@pytest.mark.parametrize("case", sorted(CASES))
def test_host_side(case, host_hip):
    env = dict(os.environ, HOST_HIP=host_hip, CHARM_HOST_THREADS="4")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], env=env, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


if __name__ == "__main__":
    sys.path[:0] = [HERE, os.path.dirname(HERE)]
    HIP = hip()
    CASES[sys.argv[1]]()
