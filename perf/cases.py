"""Performance cases of the DG time-step path.

Each case is one call sequence that a program makes through the public
binding: time steps of the benchmark workloads between two outputs (state
in, dt, N steps, conservation sums, state out), one adaptation, a reverse
sweep, a stage VJP, a batch of pointwise fluxes.  Sizes run from a few
hundred leaves or points, where latency counts, to the 2,097,152 leaves of
the Riemann box; meshes are uniform, adapted (ragged leaf counts, hanging
faces) or multi-tree; precisions are FP64, FP32 and the mixed mode.

listed() / draw(rng)   the cases
prepare(case, seed)    inputs made from the seed and the context a program keeps
run(state)             one pass
work(case)             bytes and operations a pass cannot do without
tolerance(case)        largest error another correct implementation shows
exact(case, seed)      the same outputs in FP64 by plain torch (None where a
                       value is not a computed number)
"""
import functools
import math

import numpy as np
import torch

import charm_3d_amd as CA
import charm_3d_amd.workloads as W

R_GAS = 8.31446261815324
ROOT = 1 << 19


# ------------------------------------------------------------------ cases

def listed():
    return [
        # a solver's pointwise flux calls: a few hundred point pairs
        dict(name="flux_points_small", kind="flux", points=257, flux="HLLC", precision=CA.FP64),
        # smallest time stepping: 512 leaves, periodic sine wave, reference flux of the smoke sizes
        dict(name="sine_l3_fp64", kind="steps", flow="sine", level=3, depth=0, flux="LF", limiter=False,
             precision=CA.FP64, steps=10),
        # the sine-wave benchmark in full: level 4, Lax-Friedrichs, 100 steps
        dict(name="sine_l4_fp32", kind="steps", flow="sine", level=4, depth=0, flux="LF", limiter=False,
             precision=CA.FP32, steps=100),
        # Riemann box on an adapted mesh (ragged leaf count, hanging faces), mixed precision
        dict(name="riemann_adapted_mix", kind="steps", flow="riemann", level=4, depth=2, flux="HLLC",
             limiter=True, precision=CA.FP32_MIX, steps=20),
        # Riemann box in FP64 (the benchmark's reference precision) at level 6
        dict(name="riemann_l6_fp64", kind="steps", flow="riemann", level=6, depth=0, flux="HLLC", limiter=True,
             precision=CA.FP64, steps=40),
        # the benchmark itself: level-7 Riemann box, 2,097,152 leaves, FP32
        dict(name="riemann_l7_fp32", kind="steps", flow="riemann", level=7, depth=0, flux="HLLC", limiter=True,
             precision=CA.FP32, steps=40),
        # two-species bubble on an adapted mesh: exact Riemann solver, mixture EOS, between two adaptations
        dict(name="bubble_adapted_fp32", kind="steps", flow="bubble", level=5, depth=2, flux="GODUNOV",
             limiter=True, precision=CA.FP32, steps=20),
        # reacting hot spot at its benchmark size: four species, BR2 viscous terms, diffusion, chemistry
        dict(name="hot_spot_l6_fp32", kind="hot_spot", level=6, precision=CA.FP32, br2_eta=6.0, steps=10),
        # reverse direction: gradient of the pulse objective, checkpointed
        dict(name="pulse_adjoint_l5_fp32", kind="adjoint", level=5, precision=CA.FP32, steps=40, ckpt=10),
        # one reverse stage in FP64 (reference gradients), adapted mesh
        dict(name="stage_vjp_adapted_fp64", kind="stage_vjp", level=3, depth=2, flux="HLLC", precision=CA.FP64),
        # Riemann box on 64 distorted trees (general hexahedra): 262,144 leaves
        dict(name="multi_tree_l4_fp32", kind="multi_tree", trees=4, level=4, precision=CA.FP32, flux="HLLC",
             limiter=True, steps=20),
        # one adaptation of the bubble: estimator, flags, refine / coarsen / balance, projection
        dict(name="bubble_adapt_fp32", kind="adapt", level=4, depth=2, precision=CA.FP32),
    ]


def draw(rng):
    kind = rng.choice(["flux", "steps", "steps", "steps", "steps", "hot_spot", "adjoint", "stage_vjp",
                       "multi_tree", "multi_tree", "adapt"])
    if kind == "flux":
        return dict(kind=kind, points=int(math.exp(rng.uniform(math.log(1), math.log(200000)))),
                    flux=rng.choice(["LF", "HLLC", "GODUNOV", "CD"]),
                    precision=rng.choice([CA.FP64, CA.FP32]))
    if kind == "steps":
        flow = rng.choice(["sine", "riemann", "riemann", "bubble"])
        # adapted meshes have one or two further levels about a sphere of any radius
        depth = rng.choice([0, 1, 2, 2])
        case = dict(kind=kind, flow=flow, level=rng.randint(3, 6 - depth), depth=depth,
                    steps=rng.randint(5, 30))
        if depth:
            case["radius"] = round(rng.uniform(0.15, 0.42), 4)
        if flow == "sine":
            # without a limiter the P1 scheme wants a CFL number of 0.1 away from the benchmark's settings
            case.update(flux=rng.choice(["LF", "HLLC"]), limiter=False, cfl=0.1,
                        precision=rng.choice([CA.FP64, CA.FP32, CA.FP32_MIX]))
        elif flow == "riemann":
            case.update(flux=rng.choice(["HLLC", "HLLC", "LF"]), limiter=True,
                        precision=rng.choice([CA.FP64, CA.FP32, CA.FP32_MIX]))
        else:
            case.update(flux=rng.choice(["GODUNOV", "HLLC"]), limiter=True,
                        precision=rng.choice([CA.FP64, CA.FP32]))
        return case
    if kind == "hot_spot":
        return dict(kind=kind, level=rng.randint(3, 5), precision=rng.choice([CA.FP64, CA.FP32]),
                    br2_eta=rng.choice([0.0, 6.0]), steps=rng.randint(2, 8))
    if kind == "adjoint":
        return dict(kind=kind, level=rng.randint(3, 5), precision=rng.choice([CA.FP64, CA.FP32]),
                    steps=rng.randint(5, 30), ckpt=rng.choice([0, 4, 7, 10]))
    if kind == "stage_vjp":
        return dict(kind=kind, level=rng.randint(2, 4), depth=rng.choice([1, 2]),
                    radius=round(rng.uniform(0.15, 0.42), 4), flux=rng.choice(["HLLC", "LF"]),
                    precision=rng.choice([CA.FP64, CA.FP32]))
    if kind == "multi_tree":
        return dict(kind=kind, trees=rng.randint(2, 5), level=rng.randint(2, 3),
                    precision=rng.choice([CA.FP64, CA.FP32]), flux=rng.choice(["HLLC", "LF"]),
                    limiter=True, steps=rng.randint(3, 20))
    return dict(kind="adapt", level=rng.randint(3, 4), depth=rng.choice([1, 2]),
                radius=round(rng.uniform(0.15, 0.42), 4), precision=rng.choice([CA.FP64, CA.FP32]))


# ------------------------------------------------- meshes (numpy, no library code)

def _morton(x, y, z):
    key = np.zeros(len(x), dtype=np.int64)
    for b in range(12):
        for a, v in enumerate((x, y, z)):
            key |= ((v >> b) & 1) << (3 * b + a)
    return key


def _uniform(level):
    i = np.arange(1 << level)
    x, y, z = (a.ravel() for a in np.meshgrid(i, i, i, indexing="ij"))
    order = np.argsort(_morton(x, y, z), kind="stable")
    h = ROOT >> level
    return np.stack([x[order] * h, y[order] * h, z[order] * h, np.full(len(x), level)], 1)


def _children(q):
    h = ROOT >> (q[:, 3] + 1)
    out = np.repeat(q[:, None, :], 8, axis=1)
    for c in range(8):
        for a in range(3):
            out[:, c, a] += ((c >> a) & 1) * h
    out[:, :, 3] += 1
    return out.reshape(-1, 4)


def _centres(leaves):
    h = (ROOT >> leaves[:, 3].astype(np.int64)) / ROOT
    return leaves[:, :3] / ROOT + 0.5 * h[:, None], h


@functools.lru_cache(maxsize=8)
def _leaves_of(level, depth, radius):
    """A uniform level, then `depth` levels about a sphere: leaves nearer to it
    than 3 (then 1.2) of their edges are refined, which stays 2:1."""
    q = _uniform(level)
    for d in range(depth):
        c, h = _centres(q)
        near = np.abs(np.sqrt(((c - 0.5) ** 2).sum(1)) - radius) < (3.0 - 1.8 * d) * h
        near &= q[:, 3] == level + d
        q = np.concatenate([q[~near], _children(q[near])])
    s = ROOT >> 10
    return np.ascontiguousarray(q[np.argsort(_morton(q[:, 0] // s, q[:, 1] // s, q[:, 2] // s), kind="stable")],
                                dtype=np.int32)


def _leaves(case):
    return _leaves_of(case["level"], case.get("depth", 0), case.get("radius", 0.31))


def _box_trees(n, distort=0.1):
    """n^3 trees of a unit box, vertices displaced by up to `distort` of a tree
    (within their side's plane on the box's sides)."""
    rng = np.random.default_rng(n)
    idx = np.stack(np.meshgrid(*[np.arange(n + 1)] * 3, indexing="ij"), -1)
    free = (idx > 0) & (idx < n)
    v = idx / n + np.where(free, distort / n * rng.uniform(-1, 1, idx.shape), 0.0)
    vid = np.arange((n + 1) ** 3).reshape([n + 1] * 3)
    t = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)
    t2v = np.stack([vid[t[:, 0] + (c & 1), t[:, 1] + (c >> 1 & 1), t[:, 2] + (c >> 2)] for c in range(8)], 1)
    bnd = np.full((len(t), 6), -1, np.int32)
    for f in range(6):
        bnd[t[:, f // 2] == (n - 1 if f & 1 else 0), f] = f
    return v.reshape(-1, 3), t2v.astype(np.int32), bnd, t


# ----------------------------------------------------------- flows (inputs)

# gas of the single-species flows: R / M = 1, cp = 3.5 (gamma 1.4)
_AIR = dict(m=(R_GAS,), cp=(3.5,))
# two-species bubble: gamma 1.4 / 1.67, M 0.029 / 0.004
_BUB_M, _BUB_G = (0.029, 0.004), (1.4, 1.67)
_BUBBLE = dict(m=_BUB_M, cp=tuple(g * R_GAS / ((g - 1) * m) for g, m in zip(_BUB_G, _BUB_M)))
_INLET = (0.5, 0.0, 0.0, 1.0, 1.0)


def _gas(case):
    return _BUBBLE if case.get("flow") == "bubble" or case["kind"] == "adapt" else _AIR


def _cons(rho, vel, p, gamma=1.4):
    return np.concatenate([rho[:, None] * vel, (p / (gamma - 1) + 0.5 * rho * (vel ** 2).sum(1))[:, None],
                           rho[:, None]], 1)


def _project(leaves, fn, nv):
    """FP64 L2 projection onto the P1 Taylor basis, 8 Gauss points"""
    c, h = _centres(leaves)
    u = np.zeros((len(c), nv, 4))
    for g in range(8):
        ph = np.array([(1 if g >> a & 1 else -1) * 0.5 / math.sqrt(3) for a in range(3)])
        f = fn(c + h[:, None] * ph)
        u[:, :, 0] += f / 8
        u[:, :, 1:] += 1.5 * f[:, :, None] * ph
    return u


def _flow_state(case, seed, leaves, centres=None):
    """FP64 [n][V][4] initial state of a case's flow"""
    rng = np.random.default_rng(seed)
    flow = case.get("flow", "riemann")
    if flow == "sine":
        amp, ph = rng.uniform(0.1, 0.3), rng.uniform(0, 1)

        def fn(x):
            rho = 1 + amp * np.sin(2 * np.pi * (x.sum(1) + ph))
            return _cons(rho, np.broadcast_to([1.0, 0.5, 0.25], x.shape), np.ones(len(x)))
        return _project(leaves, fn, 5)
    if flow == "bubble":
        # the adaptation keeps one density field (its leaf count is the case's); pressure and velocity vary
        c0 = 0.5 + (0.0 if case["kind"] == "adapt" else rng.uniform(-0.03, 0.03, 3))
        r0, hot = case.get("radius", 0.31), rng.uniform(0.95, 1.05)
        vel0 = rng.uniform(0.5, 1.0) * np.array([100.0, 50.0, 25.0])
        width = 3.0 / (1 << (case["level"] + case.get("depth", 0)))

        def fn(x):
            cb = 0.5 * (1 + np.tanh((r0 - np.sqrt(((x - c0) ** 2).sum(1))) / width))
            y = np.stack([1 - cb, cb], 1)
            mi = (y / np.array(_BUB_M)).sum(1)
            rho = 1.0e5 / (R_GAS * 300.0 * mi)
            cv = (y * np.array(_BUBBLE["cp"])).sum(1) - R_GAS * mi
            vel = np.broadcast_to(vel0, x.shape)
            e = cv * 300.0 * hot + 0.5 * (vel ** 2).sum(1)
            return np.concatenate([rho[:, None] * vel, (rho * e)[:, None], rho[:, None] * y], 1)
        return _project(leaves, fn, 6)
    # Riemann box: (rho, p) = (1, 1) | (0.125, 0.1) at x = 0.5, means scaled by 1 +- 1%
    c = _centres(leaves)[0] if centres is None else centres
    left = c[:, 0] < 0.5
    rho = np.where(left, 1.0, 0.125) * (1 + 0.01 * rng.uniform(-1, 1, len(c)))
    p = np.where(left, 1.0, 0.1) * (1 + 0.01 * rng.uniform(-1, 1, len(c)))
    u = np.zeros((len(c), 5, 4))
    u[:, :, 0] = _cons(rho, np.zeros((len(c), 3)), p)
    return u


def _smooth_state(leaves, seed):
    """smooth density, pressure and velocity fields (no ties of the flux's switches)"""
    ph = np.random.default_rng(seed).uniform(0, 1, (5, 3))

    def fn(x):
        f = [np.sin(2 * np.pi * ((x + p) * (1 + i % 2, 1, 1 + i // 2 % 2)).sum(1)) for i, p in enumerate(ph)]
        return _cons(1 + 0.2 * f[0], 0.3 + 0.2 * np.stack(f[1:4], 1), 1 + 0.2 * f[4])
    return _project(leaves, fn, 5)


def _pulse_state(leaves, seed):
    x0 = 0.3 + np.random.default_rng(seed).uniform(-0.05, 0.05, 3)

    def fn(x):
        rho = 1 + 0.1 * np.exp(-((x - x0) ** 2).sum(1) / 0.01)
        return _cons(rho, np.zeros((len(x), 3)), np.ones(len(x)))
    return _project(leaves, fn, 5)


_PULSE_BOX = ((0.6, 0.6, 0.6), (0.8, 0.8, 0.8))


@functools.lru_cache(maxsize=1)
def _species():
    """the hot spot's species data: (cp power series per unit mass [4][5])"""
    return [[a * R_GAS / m for a in fit] for fit, m in zip(W.c4_cp_over_r(), W.C4_M)]


def _hot_spot_state(leaves, seed):
    c0 = 0.5 + np.random.default_rng(seed).uniform(-0.05, 0.05, 3)
    y, cps = np.array(W.C4_Y), _species()
    mi = (y / np.array(W.C4_M)).sum()

    def fn(x):
        t = 300 + 1200 * np.exp(-((x - c0) ** 2).sum(1) / 0.01)
        cp = sum(y[i] * sum(c * t ** k for k, c in enumerate(cps[i])) for i in range(4))
        rho = 101325.0 / (R_GAS * t * mi)
        out = np.zeros((len(x), 8))
        out[:, 3] = rho * (cp - R_GAS * mi) * t
        out[:, 4:] = rho[:, None] * y
        return out
    return _project(leaves, fn, 8)


_HOT_DT = 0.3 / 1500.0            # CFL 0.3 over the sound speed of the hottest gas, times h


def _flux_rows(case, seed):
    """point pairs (r, u, v, w, p, c) across moderate jumps, random unit normals"""
    rng = np.random.default_rng(seed)
    n = case["points"]
    rows = []
    for _ in range(2):
        rows.append(np.concatenate([rng.uniform(0.1, 1.2, (n, 1)), rng.uniform(-0.6, 0.6, (n, 3)),
                                    rng.uniform(0.1, 1.2, (n, 1)), np.ones((n, 1))], 1))
    nn = rng.normal(size=(n, 3))
    return rows[0], rows[1], nn / np.linalg.norm(nn, axis=1, keepdims=True)


# ---------------------------------------------------------- prepare / run

def _config(case):
    prec = case["precision"]
    gas = _gas(case)
    kind = case["kind"]
    if kind == "hot_spot":
        return W.c4_config(prec, visc_br2_eta=case["br2_eta"])
    kw = dict(precision=prec, model="NS", flux=case.get("flux", "HLLC"), limiter=case.get("limiter", False),
              comp_m=gas["m"], comp_cp=gas["cp"], bnd=("OUTLET",) * 6, cfl=case.get("cfl", 0.3))
    if case.get("flow") == "sine":
        kw["bnd"] = ("PERIODIC",) * 6
    if gas is _BUBBLE:
        kw["eos"] = "MIX"
    if kind == "adapt":
        kw.update(flux="GODUNOV", limiter=True, max_err=0.04, min_level=case["level"] - 1,
                  max_level=case["level"] + case["depth"] + 1)
    if kind in ("adjoint", "stage_vjp"):
        kw.update(bnd=("INLET",) + ("OUTLET",) * 5, bnd_param=[_INLET] + [None] * 5, cfl=0.1)
    return CA.make_config(**kw)


def _gm_centres(case):
    """leaf centres and smallest extent of the multi-tree case, tree by tree"""
    g = _gm_geometry(case["trees"], case["level"])
    return g["c"], g["dh"].min()


def prepare(case, seed):
    kind = case["kind"]
    cfg = _config(case)
    ctx = CA.GpuContext(cfg)
    st = dict(case=case, ctx=ctx)
    if kind == "flux":
        st["args"] = _flux_rows(case, seed)
        return st
    if kind == "multi_tree":
        v, t2v, bnd, _ = _box_trees(case["trees"])
        st["mesh"] = CA.GMesh(v, t2v, bnd, case["level"])
        ctx.upload_gmesh(st["mesh"])
        c, dh = _gm_centres(case)
        st["u0"] = _flow_state(case, seed, None, c)
        st["dt"] = _gm_dt(st["u0"], dh)
        return st
    leaves = _leaves(case)
    per = (case.get("flow") == "sine",) * 3
    chunks = CA.recommended_chunks(cfg)
    st["mesh"] = CA.Forest.from_leaves(leaves, per).flatten(*chunks)
    ctx.upload_mesh(st["mesh"])
    if kind == "steps":
        st["u0"] = _flow_state(case, seed, leaves)
    elif kind == "hot_spot":
        st["u0"], st["dt"] = _hot_spot_state(leaves, seed), _HOT_DT / (1 << case["level"])
    elif kind == "adjoint":
        st["u0"], st["dt"] = _pulse_state(leaves, seed), 0.1 / (1 << case["level"]) / 1.7
    elif kind == "stage_vjp":
        st["u0"] = _smooth_state(leaves, seed)
        st["x"] = np.random.default_rng(seed + 1).normal(size=st["u0"].shape)
        st["dt"] = 0.1 / (1 << (case["level"] + case["depth"])) / 1.7
    else:
        st.update(u0=_flow_state(dict(case, flow="bubble"), seed, leaves), leaves=leaves, chunks=chunks)
    return st


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "flux":
        return ctx.flux_batch(case["flux"], *state["args"])
    if kind == "steps":
        # one output interval of a run: CFL step, steps, conservation log, solution
        ctx.set_state(state["u0"])
        dt = ctx.get_dt(1)
        ctx.run(dt, case["steps"])
        return dict(dt=dt, sums=ctx.conservation_sums(), state=ctx.get_state())
    if kind in ("hot_spot", "multi_tree"):
        ctx.set_state(state["u0"])
        ctx.run(state["dt"], case["steps"])
        return ctx.get_state()
    if kind == "adjoint":
        ctx.set_state(state["u0"])
        j, grad, theta, _, _ = ctx.adjoint(state["dt"], case["steps"], *_PULSE_BOX, ckpt=case["ckpt"], theta_face=0)
        return dict(j=j, grad=grad, theta=theta)
    if kind == "stage_vjp":
        return ctx.stage_vjp(state["dt"], state["u0"], state["x"])
    # one adaptation, from the state on the old mesh to the projected one
    cfg = ctx.cfg
    ctx.upload_mesh(state["mesh"])
    ctx.set_state(state["u0"])
    err2, rho = ctx.amr_indicator()
    flags = CA.amr_flags(state["leaves"], err2, rho, cfg.max_err, cfg.min_level, cfg.max_level)
    forest = CA.Forest.from_leaves(state["leaves"])
    amap = forest.adapt(flags, cfg.max_level, cfg.min_level)
    ctx.remesh(forest.flatten(*state["chunks"]), amap)
    return dict(err2=err2, rho=rho, leaves=forest.leaves(), state=ctx.get_state())


# -------------------------------------------------------- work, tolerance

def work(case):
    """The caller's FP64 arrays read and written once, and the operations of
    the scheme: per stage the fluxes at the six points of three faces and
    the eight volume points of each leaf."""
    kind = case["kind"]
    if kind == "flux":
        n = case["points"]
        return dict(bytes=8 * n * (2 * 6 + 3 + 5), flops=150 * n)
    n = case["trees"] ** 3 * 8 ** case["level"] if kind == "multi_tree" else len(_leaves(case))
    nv = 8 if kind == "hot_spot" else 4 + len(_gas(case)["m"])
    io = 2 * n * nv * 4 * 8
    # two traces, two states, a flux and its moments per face point; a trace, a state and three fluxes per volume point
    stage = n * (18 * (18 * nv + 150) + 8 * (6 * nv + 75) + 8 * nv)
    if kind == "adapt":
        return dict(bytes=io + 2 * 8 * n, flops=200 * n)
    if kind == "stage_vjp":
        return dict(bytes=io // 2 * 3, flops=3 * stage)
    # viscous terms, diffusion and chemistry: about two more evaluations; a reverse step: about three
    times = {"hot_spot": 3, "adjoint": 4}.get(kind, 1)
    return dict(bytes=io, flops=3 * case["steps"] * times * stage)


def tolerance(case):
    """Relative 2-norm errors, four times the largest that the paths show
    against the FP64 evaluation over these ranges.  FP32 time steps gather
    rounding over up to 100 steps (3.9e-6); the limiter's switches at the
    shock carry it further in the Riemann box (4.0e-6 after 40 steps at level
    7; mixed mode 2.5e-7).  FP64 is rounding (5e-14), except that the exact
    Riemann solver stops its Newton at a velocity residual of 1e-5 (3.3e-12)
    and the adjoint starts from a state at rest, on the flux's switches
    (2.5e-11)."""
    kind, prec = case["kind"], case["precision"]
    if kind == "adapt":
        # leaf sets are whole numbers; the estimator and projection run in FP64 on the stored state
        return {"rel": 1e-6 if prec == CA.FP32 else 1e-13, "differ": 0.0}
    if prec == CA.FP64:
        return {"rel": 1e-10 if kind == "adjoint" or case.get("flux") == "GODUNOV" else 1e-12}
    if prec == CA.FP32_MIX:
        return {"rel": 1e-6}
    return {"rel": {"flux": 1.5e-6, "hot_spot": 8e-7, "adjoint": 6.5e-6, "stage_vjp": 2.5e-6}.get(kind, 1.6e-5)}


# ------------------------------------------------ FP64 reference (plain torch)
#
# A mesh is face groups (side-0 / side-1 leaves, basis values of the six
# points on either side, weights, side-0 normal; boundary groups name a slot)
# and per-leaf volume points, 1/dh, A^-1, vertex basis values and basis
# means.  Fields are [..][n] tensors, a state is u[V][4][n].

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev())


_GP1 = np.array([-1 / 3, 1 / 6, -1 / 3, 1 / 3, -1 / 6, 1 / 3])
_GP2 = np.array([-1 / 3, -1 / 3, 1 / 6, -1 / 6, 1 / 3, 1 / 3])


def _basis(axis, pn, q1, q2):
    """[3][6] basis values of the face points: pn along the axis, q1 < q2 the others"""
    t1, t2 = [a for a in range(3) if a != axis]
    b = np.zeros((3, 6))
    b[axis], b[t1], b[t2] = pn, q1, q2
    return _t(b)[:, :, None]


def _octree(leaves, periodic):
    """face groups and leaf data of a 2:1 octree on the unit cube"""
    q = leaves.astype(np.int64)
    unit = ROOT >> 10
    x, lev = q[:, :3] // unit, q[:, 3]
    size = 1024 >> lev
    h = size / 1024.0

    def code(lv, p):
        return ((lv * 1024 + p[:, 0]) * 1024 + p[:, 1]) * 1024 + p[:, 2]
    keys = code(lev, x)
    order = np.argsort(keys)

    def find(lv, p):
        k = code(lv, p)
        pos = np.minimum(np.searchsorted(keys[order], k), len(keys) - 1)
        return np.where(keys[order][pos] == k, order[pos], -1)

    groups, nbr = [], []
    for a in range(3):
        t1, t2 = [b for b in range(3) if b != a]
        for side in (0, 1):
            p = x.copy()
            p[:, a] += np.where(side, size, -size)
            out = (p[:, a] < 0) | (p[:, a] >= 1024)
            if periodic:
                p[:, a] %= 1024
                out[:] = False
            same = np.where(out, -1, find(lev, p))
            big_size = size * 2
            bp = p // big_size[:, None] * big_size[:, None]
            big = np.where(out | (same >= 0), -1, find(lev - 1, bp))
            sub = (p[:, t1] // size & 1) + 2 * (p[:, t2] // size & 1)
            s = 0.5 if side else -0.5
            if side:
                e = np.flatnonzero(same >= 0)
                groups.append((e, same[e], _basis(a, s, _GP1, _GP2), _basis(a, -s, _GP1, _GP2), a, 1.0, None, 1.0, 1.0))
            for j in range(4):
                e = np.flatnonzero((big >= 0) & (sub == j))
                d1, d2 = (0.25 if j & 1 else -0.25), (0.25 if j & 2 else -0.25)
                groups.append((e, big[e], _basis(a, s, _GP1, _GP2),
                               _basis(a, -s, d1 + _GP1 / 2, d2 + _GP2 / 2), a, 2.0 * s, None, 1.0, 0.25))
            e = np.flatnonzero(out)
            groups.append((e, None, _basis(a, s, _GP1, _GP2), None, a, 2.0 * s, 2 * a + side, 1.0, 0.0))
    fg = []
    for e0, e1, b0, b1, a, sgn, slot, w0, w1 in groups:
        if len(e0) == 0:
            continue
        n = torch.zeros(3, 1, 1, dtype=torch.float64, device=_dev())
        n[a] = sgn
        fg.append(dict(e0=_t(e0), e1=None if e1 is None else _t(e1), b0=b0, b1=b1, slot=slot, axis=a, n=n,
                       w=_t(np.broadcast_to(h[e0] ** 2 / 6, (6, len(e0))).copy()), dir=2 * a + (1 if sgn > 0 else 0),
                       share=(w0, w1)))
    s3 = 0.5 / math.sqrt(3)
    vb = np.array([[(s3 if g >> a & 1 else -s3) for g in range(8)] for a in range(3)])
    vv = np.array([[(0.5 if g >> a & 1 else -0.5) for g in range(8)] for a in range(3)])
    ai = torch.zeros(4, 4, len(h), dtype=torch.float64, device=_dev())
    for k, f in enumerate((1.0, 12.0, 12.0, 12.0)):
        ai[k, k] = f * _t(8.0 ** lev)
    hh = _t(h)
    return dict(n=len(h), faces=fg, vb=_t(vb)[:, :, None], vw=(hh ** 3 / 8).expand(8, -1), dhi=(1 / hh).expand(3, -1),
                ai=ai, vert=_t(vv)[:, :, None], mb=torch.zeros(3, 1, dtype=torch.float64, device=_dev()), h=hh,
                vol=hh ** 3, lev=_t(lev), x=_t(x))


@functools.lru_cache(maxsize=2)
def _gm_geometry(ntree, level):
    """trilinear leaf geometry of the box of trees, leaves tree by tree in
    Morton order: corners [n][8][3], centre, bounding-box extents"""
    v, t2v, _, t = _box_trees(ntree)
    q = _uniform(level)[:, :3] // (ROOT >> level)
    side = 1 << level
    pos = (t[:, None, :] * side + q[None, :, :]).reshape(-1, 3)
    tv = np.repeat(v[t2v], len(q), axis=0)
    ref = np.tile(q, (len(t), 1))

    def point(off):
        r = (ref + off) / side
        out = np.zeros((len(ref), 3))
        for c in range(8):
            w = np.ones(len(ref))
            for a in range(3):
                w = w * (r[:, a] if c >> a & 1 else 1 - r[:, a])
            out += w[:, None] * tv[:, c]
        return out
    corners = np.stack([point(np.array([c & 1, c >> 1 & 1, c >> 2])) for c in range(8)], 1)
    return dict(corners=corners, c=point(0.5), dh=corners.max(1) - corners.min(1), pos=pos)


def _gm_mesh(ntree, level):
    """face groups and leaf data of the distorted box (two triangles per face)"""
    g = _gm_geometry(ntree, level)
    cor, c, dh, pos = g["corners"], g["c"], g["dh"], g["pos"]
    nn = ntree << level
    grid = np.zeros((nn, nn, nn), dtype=np.int64)
    grid[pos[:, 0], pos[:, 1], pos[:, 2]] = np.arange(len(pos))
    fg = []
    for a in range(3):
        t1, t2 = [b for b in range(3) if b != a]
        for side in (0, 1):
            p = pos.copy()
            p[:, a] += 1 if side else -1
            out = (p[:, a] < 0) | (p[:, a] >= nn)
            for bnd in (False, True):
                if not bnd and not side:
                    continue
                e0 = np.flatnonzero(out == bnd)
                if len(e0) == 0:
                    continue
                fc = [(side << a) + (i << t1) + (j << t2) for j in (0, 1) for i in (0, 1)]
                x = cor[e0][:, fc]
                nrm = np.cross(x[:, 1] - x[:, 0], x[:, 2] - x[:, 0])
                nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
                nrm *= np.sign((nrm * (x.mean(1) - c[e0])).sum(1))[:, None]
                pts, wj = [], []
                for i in range(2):
                    d1, d2 = x[:, i] - x[:, i + 2], x[:, i + 1] - x[:, i + 2]
                    area = np.linalg.norm(np.cross(d1, d2), axis=1) / 6
                    for wa, wb in ((2 / 3, 1 / 6), (1 / 6, 2 / 3), (1 / 6, 1 / 6)):
                        pts.append(wa * d1 + wb * d2 + x[:, i + 2])
                        wj.append(area)
                pts = np.stack(pts, 1)

                def rel(e):
                    return _t(((pts - c[e][:, None]) / dh[e][:, None]).transpose(2, 1, 0))
                e1 = None if bnd else grid[tuple(p[e0].T)]
                fg.append(dict(e0=_t(e0), e1=None if bnd else _t(e1), b0=rel(e0), b1=None if bnd else rel(e1),
                               slot=2 * a + side if bnd else None, axis=a, n=_t(nrm.T.copy())[:, None, :],
                               w=_t(np.stack(wj)), dir=2 * a + side, share=(1.0, 1.0)))
    s3 = 1 / math.sqrt(3)
    vb, vw = [], []
    for k in range(8):
        r = [s3 if k >> a & 1 else -s3 for a in range(3)]
        gp, jac = 0.0, [0.0, 0.0, 0.0]
        for q in range(8):
            w = [1 + r[a] if q >> a & 1 else 1 - r[a] for a in range(3)]
            d = [1.0 if q >> a & 1 else -1.0 for a in range(3)]
            gp = gp + w[0] * w[1] * w[2] / 8 * cor[:, q]
            for a in range(3):
                b0, b1 = [b for b in range(3) if b != a]
                jac[a] = jac[a] + d[a] * w[b0] * w[b1] / 8 * cor[:, q]
        vb.append((gp - c) / dh)
        vw.append((jac[0] * np.cross(jac[1], jac[2])).sum(1))
    vb, vw = np.stack(vb, 1), np.stack(vw, 1)
    phi = np.concatenate([np.ones(vb.shape[:2] + (1,)), vb], 2)
    ai = np.linalg.inv(np.einsum("ng,ngi,ngj->nij", vw, phi, phi))
    vol = vw.sum(1)
    return dict(n=len(c), faces=fg, vb=_t(vb.transpose(2, 1, 0)), vw=_t(vw.T), dhi=_t(1 / dh.T), ai=_t(ai.transpose(1, 2, 0)),
                vert=_t(((cor - c[:, None]) / dh[:, None]).transpose(2, 1, 0)),
                mb=_t(((vw[:, :, None] * vb).sum(1) / vol[:, None]).T), vol=_t(vol))


class _Gas:
    """EOS of constant or power-series cp; T by Newton for the latter"""

    def __init__(self, m, cp):
        self.m = [float(x) for x in m]
        self.cp = [list(c) if isinstance(c, (list, tuple)) else [float(c)] for c in cp]
        self.poly = any(len(c) > 1 for c in self.cp)

    def prim(self, u):
        rho = u[4:].sum(0)
        s = dict(r=rho, v=[u[d] / rho for d in range(3)], c=[(x / rho).clamp(0.0, 1.0) for x in u[4:]], E=u[3])
        s["e"] = u[3] / rho - 0.5 * sum(v * v for v in s["v"])
        mi = sum(c / m for c, m in zip(s["c"], self.m))
        a = [sum(c * k[j] for c, k in zip(s["c"], self.cp) if j < len(k)) for j in range(max(map(len, self.cp)))]
        if self.poly:
            t = torch.full_like(rho, 600.0)
            for _ in range(9):
                cp, dcp = a[-1], torch.zeros_like(rho)
                for k in range(len(a) - 2, -1, -1):
                    dcp = dcp * t + cp
                    cp = cp * t + a[k]
                t = t - ((cp - R_GAS * mi) * t - s["e"]) / (cp - R_GAS * mi + dcp * t)
            cp = sum(x * t ** k for k, x in enumerate(a))
        else:
            cp = a[0]
        cv = cp - R_GAS * mi
        s.update(gam=cp / cv, cv=cv, m=1 / mi, T=s["e"] / cv)
        s["p"] = rho * s["e"] * (s["gam"] - 1)
        s["cz"] = torch.sqrt(s["gam"] * s["p"] / rho)
        return s


def _exterior(s, bc, slot, n):
    """boundary state: transmissive, or an inlet's (u, T, p)"""
    if bc is None or bc[slot] is None:
        return s
    u, v, w, t, p = bc[slot]
    one = torch.ones_like(s["r"])
    o = dict(s, v=[u * one, v * one, w * one], p=p * one, T=t * one)
    o["r"] = o["p"] * s["m"] / (R_GAS * o["T"])
    o["e"] = o["p"] / (o["r"] * (s["gam"] - 1))
    o["E"] = o["r"] * (o["e"] + 0.5 * sum(x * x for x in o["v"]))
    o["cz"] = torch.sqrt(s["gam"] * o["p"] / o["r"])
    return o


def _flux(kind, L, Rt, n):
    """flux along n: [V] list of tensors"""
    un = [sum(s["v"][d] * n[d] for d in range(3)) for s in (L, Rt)]
    if kind in ("LF", "CD"):
        al = torch.maximum(un[0].abs() + L["cz"], un[1].abs() + Rt["cz"]) if kind == "LF" else 0.0
        out = []
        for d in range(3):
            f = [s["r"] * x * s["v"][d] + s["p"] * n[d] for s, x in zip((L, Rt), un)]
            out.append(0.5 * (f[0] + f[1] - al * (Rt["r"] * Rt["v"][d] - L["r"] * L["v"][d])))
        out.append(0.5 * ((L["E"] + L["p"]) * un[0] + (Rt["E"] + Rt["p"]) * un[1] - al * (Rt["E"] - L["E"])))
        for a, b in zip(L["c"], Rt["c"]):
            out.append(0.5 * (L["r"] * un[0] * a + Rt["r"] * un[1] * b - al * (Rt["r"] * b - L["r"] * a)))
        return out
    if kind == "GODUNOV":
        return _exact_riemann(L, Rt, un, n)
    pv = 0.5 * (L["p"] + Rt["p"]) - 0.125 * (un[1] - un[0]) * (L["r"] + Rt["r"]) * (L["cz"] + Rt["cz"])
    ps = pv.clamp(min=0.0)
    q = []
    for s in (L, Rt):
        x = 1 + (s["gam"] + 1) / (2 * s["gam"]) * (ps / s["p"] - 1)
        shock = ps > s["p"]
        q.append(torch.where(shock, torch.sqrt(torch.where(shock, x, torch.ones_like(x))), torch.ones_like(x)))
    s0, s1 = un[0] - L["cz"] * q[0], un[1] + Rt["cz"] * q[1]
    sl, sr = torch.minimum(s0, s1), torch.maximum(s0, s1)
    al, ar = L["r"] * (sl - un[0]), Rt["r"] * (sr - un[1])
    ss = (Rt["p"] - L["p"] + un[0] * al - un[1] * ar) / (al - ar)
    ss = torch.minimum(torch.maximum(ss, sl), sr)
    sup = (sl >= 0) | (sr <= 0)
    left = (sl >= 0) | (~(sr <= 0) & (ss >= 0))

    def pick(a, b):
        return torch.where(left, a, b)
    r, p, E, u, sk = pick(L["r"], Rt["r"]), pick(L["p"], Rt["p"]), pick(L["E"], Rt["E"]), pick(*un), pick(sl, sr)
    inv = 1 / torch.where(sup, torch.ones_like(sk), sk - ss)
    pk = p + r * (sk - u) * (ss - u)
    out = []
    for d in range(3):
        v = pick(L["v"][d], Rt["v"][d])
        star = (ss * ((sk - u) * r * v - p * n[d]) + sk * pk * n[d]) * inv
        out.append(torch.where(sup, r * u * v + p * n[d], star))
    out.append(torch.where(sup, (E + p) * u, (ss * (sk * E - (E + p) * u) + sk * pk * ss) * inv))
    for a, b in zip(L["c"], Rt["c"]):
        c = pick(a, b)
        out.append(torch.where(sup, r * u * c, ss * (sk - u) * r * c * inv))
    return out


def _exact_riemann(L, Rt, un, n):
    """exact solver with one gamma per side: Newton for p*, sampled at rest"""
    side = [dict(r=s["r"], p=s["p"], u=x, c=s["cz"], g=s["gam"]) for s, x in zip((L, Rt), un)]

    def curve(s, p):
        g = s["g"]
        root = torch.sqrt(s["p"] * s["r"] * (0.5 * (g + 1) * p / s["p"] + 0.5 * (g - 1)))
        fs = (p - s["p"]) / root
        dfs = 1 / root - 0.25 * (p - s["p"]) * s["r"] * (g + 1) / root ** 3
        x = (p / s["p"]) ** (0.5 * (g - 1) / g)
        fr = 2 * s["c"] / (g - 1) * (x - 1)
        dfr = s["c"] * x / (g * p)
        sh = p > s["p"]
        return torch.where(sh, fs, fr), torch.where(sh, dfs, dfr)
    a, b = side
    z = [s["r"] * s["c"] for s in side]
    p = (a["p"] * z[1] + b["p"] * z[0] + (a["u"] - b["u"]) * z[0] * z[1]) / (z[0] + z[1])
    for _ in range(12):
        p = p.clamp(min=1e-9)
        (f0, d0), (f1, d1) = curve(a, p), curve(b, p)
        p = p + (a["u"] - b["u"] - f0 - f1) / (d0 + d1)
    us = 0.5 * (a["u"] - curve(a, p)[0] + b["u"] + curve(b, p)[0])
    left = us >= 0

    def pick(i, j):
        return torch.where(left, i, j)
    sg = torch.where(left, 1.0, -1.0).to(p.dtype)
    r, pk, u, c, g = (pick(a[k], b[k]) for k in ("r", "p", "u", "c", "g"))
    u, ust = sg * u, sg * us                         # mirrored so that the wave runs to -x
    ratio = p / pk
    shock = ratio > 1
    m2 = torch.sqrt((g + 1) / (2 * g) * ratio + (g - 1) / (2 * g))
    rs_sh = r * (ratio * (g + 1) + (g - 1)) / (ratio * (g - 1) + (g + 1))
    rs_ra = r * ratio ** (1 / g)
    cs = c * ratio ** (0.5 * (g - 1) / g)
    head = torch.where(shock, u - c * m2, u - c)
    tail = torch.where(shock, u - c * m2, ust - cs)
    ufan = 2 / (g + 1) * (c + 0.5 * (g - 1) * u)
    rfan = r * (ufan / c).clamp(min=1e-12) ** (2 / (g - 1))
    pfan = pk * (ufan / c).clamp(min=1e-12) ** (2 * g / (g - 1))
    ro = torch.where(head >= 0, r, torch.where(tail <= 0, torch.where(shock, rs_sh, rs_ra), rfan))
    uo = sg * torch.where(head >= 0, u, torch.where(tail <= 0, ust, ufan))
    po = torch.where(head >= 0, pk, torch.where(tail <= 0, p, pfan))
    vel = [pick(*[s["v"][d] + (uo - x) * n[d] for s, x in zip((L, Rt), un)]) for d in range(3)]
    E = po / (g - 1) + 0.5 * ro * sum(v * v for v in vel)
    out = [ro * uo * vel[d] + po * n[d] for d in range(3)] + [(E + po) * uo]
    return out + [ro * uo * pick(x, y) for x, y in zip(L["c"], Rt["c"])]


def _trace(u, e, b):
    """[V][points][F] values of u at basis values b for leaves e (None: all)"""
    w = u if e is None else u[:, :, e]
    return w[:, 0, None] + b[0] * w[:, 1, None] + b[1] * w[:, 2, None] + b[2] * w[:, 3, None]


def _moments(q, b, w):
    """[V][4][F]: sum over the points of q (1, b) w"""
    qw = torch.stack(torch.broadcast_tensors(*q)) * w
    return torch.stack([qw.sum(1)] + [(qw * b[d]).sum(1) for d in range(3)], 1)


def _residual(mesh, gas, flux, bc, u):
    res = torch.zeros_like(u)
    for f in mesh["faces"]:
        L = gas.prim(_trace(u, f["e0"], f["b0"]))
        Rt = _exterior(L, bc, f["slot"], f["n"]) if f["e1"] is None else gas.prim(_trace(u, f["e1"], f["b1"]))
        q = _flux(flux, L, Rt, f["n"])
        res = res.index_add(2, f["e0"], _moments(q, f["b0"], f["w"]))
        if f["e1"] is not None:
            res = res.index_add(2, f["e1"], -_moments(q, f["b1"], f["w"]))
    s = gas.prim(_trace(u, None, mesh["vb"]))
    rows = []
    for d in range(3):
        f = [s["r"] * s["v"][d] * s["v"][j] + (s["p"] if j == d else 0.0) for j in range(3)]
        f.append((s["E"] + s["p"]) * s["v"][d])
        f += [s["r"] * s["v"][d] * c for c in s["c"]]
        rows.append((torch.stack(f) * (mesh["vw"] * mesh["dhi"][d])).sum(1))
    return res - torch.stack([torch.zeros_like(rows[0])] + rows, 1)


def _solve(mesh, res):
    return torch.einsum("kjn,vjn->vkn", mesh["ai"], res)


def _limit(mesh, gas, bc, u):
    """Barth-Jespersen over the vertices, neighbour means per face direction"""
    mean = u[:, 0] + sum(mesh["mb"][d] * u[:, 1 + d] for d in range(3))
    nb = torch.zeros((6,) + mean.shape, dtype=u.dtype, device=u.device)
    for f in mesh["faces"]:
        if f["e1"] is None:
            nb[f["dir"]].index_add_(1, f["e0"], mean[:, f["e0"]])       # transmissive: its own mean
            continue
        nb[f["dir"]].index_add_(1, f["e0"], f["share"][0] * mean[:, f["e1"]])
        nb[f["dir"] ^ 1].index_add_(1, f["e1"], f["share"][1] * mean[:, f["e0"]])
    hi, lo = torch.maximum(mean, nb.amax(0)), torch.minimum(mean, nb.amin(0))
    df = _trace(u, None, mesh["vert"]) - mean[:, None]
    up, dn = df.amax(1), -df.amin(1)
    one = torch.ones_like(mean)
    psi = torch.where(up > 1e-12, torch.minimum(one, (hi - mean) / up.clamp(min=1e-12)), one)
    psi = torch.where(dn > 1e-12, torch.minimum(psi, (mean - lo) / dn.clamp(min=1e-12)), psi)
    return torch.cat([u[:, :1], u[:, 1:] * psi[:, None]], 1)


def _step(mesh, gas, flux, bc, limiter, u, dt, source=None, stages=False):
    """one SSP-RK3 step; source(u) -> (u after chemistry, extra integrals)"""
    w, old = u, []
    for combine in (None, (0.25, 0.75), (2 / 3, 1 / 3)):
        x, extra = (w, 0.0) if source is None else source(w)
        old.append(x)
        w = x - dt * _solve(mesh, _residual(mesh, gas, flux, bc, x) + extra)
        if limiter:
            w = _limit(mesh, gas, bc, w)
        if combine is not None:
            w = combine[0] * w + combine[1] * u
    return (w, old) if stages else w


def _to(u):
    return _t(u).permute(1, 2, 0).contiguous()


def _from(u):
    return u.permute(2, 0, 1).contiguous().cpu().numpy()


# viscous, diffusion and chemistry terms of the hot spot (uniform octree)

class _HotSpot:
    def __init__(self, mesh, gas, eta, dt):
        self.mesh, self.gas, self.eta, self.dt = mesh, gas, eta, dt
        self.tr = []
        for i in range(4):
            ml0, ts = W.C4_ML[i]
            cp0 = sum(c * 273.0 ** k for k, c in enumerate(gas.cp[i]))
            self.tr.append((ml0, ml0 * cp0 / 0.72, ts))

    def enthalpy(self, i, t):
        return W.C4_H0[i] + sum(c * (t ** (k + 1) - 298.15 ** (k + 1)) / (k + 1) for k, c in enumerate(self.gas.cp[i]))

    def transport(self, s):
        mu = kt = den = 0.0
        for (ml0, kp0, ts), c, m in zip(self.tr, s["c"], self.gas.m):
            f = (s["T"] / 273.0) ** 1.5 * (273.0 + ts) / (s["T"] + ts)
            den, mu, kt = den + c / m, mu + c / m * ml0 * f, kt + c * kp0 * f
        return mu / den, kt

    def diffusion(self, s):
        x = [c / m for c, m in zip(s["c"], self.gas.m)]
        tot = sum(x)
        x = [v / tot for v in x]
        out = []
        for i, (si, ei) in enumerate(W.C4_LJ):
            acc = 0.0
            for j, (sj, ej) in enumerate(W.C4_LJ):
                if i == j:
                    continue
                td = s["T"] / math.sqrt(ei * ej)
                wd = (1.06036 / td ** 0.1561 + 0.1930 * torch.exp(-0.47635 * td) + 1.03587 * torch.exp(-1.52996 * td)
                      + 1.76474 * torch.exp(-3.89411 * td))
                dij = (2.628e-7 * math.sqrt(0.5 * (1 / (1000 * self.gas.m[i]) + 1 / (1000 * self.gas.m[j])))
                       * s["T"] ** 1.5 / (s["p"] / 101325.0 * (0.5 * (si + sj)) ** 2 * wd))
                acc = acc + x[j] / dij
            out.append((1 - x[i]) / acc)
        return out

    def chemistry(self, u):
        """2 H2 + O2 -> 2 H2O on the cell means, two semi-implicit passes"""
        s = self.gas.prim(u[:, 0])
        k = W.C4_A * torch.exp(-15000.0 / s["T"])
        c = [u[4 + i, 0] / self.gas.m[i] for i in range(4)]
        ch = list(c)
        for _ in range(2):
            h2, o2 = 0.5 * (ch[0] + c[0]), 0.5 * (ch[1] + c[1])
            phi = [2 * k * h2 * o2, k * h2 * h2, 0 * k, 0 * k]
            psi = [0 * k, 0 * k, 2 * k * h2 * h2 * o2, 0 * k]
            for i in range(4):
                y = self.dt * phi[i]
                ch[i] = (c[i] + self.dt * psi[i] * (1 + 0.5 * y)) / (1 + y + 0.5 * y * y)
        w = k * ch[0] ** 2 * ch[1]
        rate = [-2 * w, -w, 2 * w, 0 * w]
        heat = sum(rate[i] * self.gas.m[i] * self.enthalpy(i, s["T"]) for i in range(4))
        out = u.clone()
        for i in range(4):
            out[4 + i] = 0.0
            out[4 + i, 0] = ch[i] * self.gas.m[i]
        return out, heat

    def terms(self, mu, kt, dm, v, t, r, c, n):
        """tau (xx yy zz xy xz yz) of v along n, and k T + sum h rho D Y along n"""
        lp, lm = 4 / 3 * mu, -2 / 3 * mu
        q = [(lp if d == 0 else lm) * v[0] * n[0] + (lp if d == 1 else lm) * v[1] * n[1]
             + (lp if d == 2 else lm) * v[2] * n[2] for d in range(3)]
        q += [mu * (v[0] * n[1] + v[1] * n[0]), mu * (v[2] * n[0] + v[0] * n[2]), mu * (v[2] * n[1] + v[1] * n[2])]
        heat = kt * t + sum(self.enthalpy(i, t) * r * dm[i] * c[i] for i in range(4))
        return q + [-heat * n[d] for d in range(3)]

    def __call__(self, u):
        x, heat = self.chemistry(u)
        mesh = self.mesh
        dco = self.diffusion(self.gas.prim(x[:, 0]))
        aux = torch.zeros(9, 4, mesh["n"], dtype=u.dtype, device=u.device)
        own = torch.zeros_like(aux)
        s = self.gas.prim(_trace(x, None, mesh["vb"]))
        mu, kt = self.transport(s)
        wd = mesh["vw"] * mesh["dhi"][0]
        for d in range(3):
            n = [1.0 if a == d else 0.0 for a in range(3)]
            vol = self.terms(mu, kt, dco, s["v"], s["T"], s["r"], s["c"], n)
            vol = (torch.stack(torch.broadcast_tensors(*[torch.as_tensor(q, device=u.device) + 0 * mu for q in vol])) * wd).sum(1)
            aux[:, 1 + d] -= vol
        own += aux
        lifts = []
        for f in mesh["faces"]:
            n = f["n"]
            L = self.gas.prim(_trace(x, f["e0"], f["b0"]))
            ml, kl = self.transport(L)
            if f["e1"] is None:
                q = self.terms(ml, kl, [c[f["e0"]] for c in dco], L["v"], L["T"], L["r"], L["c"], n)
                m = _moments(q, f["b0"], f["w"])
                aux.index_add_(2, f["e0"], m)
                own.index_add_(2, f["e0"], m)
                lifts.append(None)
                continue
            Rt = self.gas.prim(_trace(x, f["e1"], f["b1"]))
            mr, kr = self.transport(Rt)
            dm = [0.5 * (c[f["e0"]] + c[f["e1"]]) for c in dco]
            mu, kt = 0.5 * (ml + mr), 0.5 * (kl + kr)
            avg = self.terms(mu, kt, dm, [0.5 * (a + b) for a, b in zip(L["v"], Rt["v"])], 0.5 * (L["T"] + Rt["T"]),
                             0.5 * (L["r"] + Rt["r"]), [0.5 * (a + b) for a, b in zip(L["c"], Rt["c"])], n)
            pair = []
            for sgn, e, b, side in ((1, f["e0"], f["b0"], L), (-1, f["e1"], f["b1"], Rt)):
                ma = sgn * _moments(avg, b, f["w"])
                mo = sgn * _moments(self.terms(mu, kt, dm, side["v"], side["T"], side["r"], side["c"], n), b, f["w"])
                aux.index_add_(2, e, ma)
                own.index_add_(2, e, mo)
                pair.append(torch.einsum("kjn,vjn->vkn", mesh["ai"][:, :, e], ma - mo))
            lifts.append(pair)
        aux, own = _solve(mesh, aux), _solve(mesh, own)
        # viscous integrals of ru rv rw re
        out = torch.zeros_like(u)
        tau = _trace(aux, None, mesh["vb"])
        row = [[tau[0], tau[3], tau[4]], [tau[3], tau[1], tau[5]], [tau[4], tau[5], tau[2]]]
        phi = [torch.ones_like(mesh["vb"][0])] + [mesh["vb"][d] for d in range(3)]
        for d in range(3):
            for j in range(3):
                out[j, 1 + d] += (row[j][d] * wd).sum(0)
            out[3, 1 + d] += (sum(row[d][j] * s["v"][j] for j in range(3)) * wd).sum(0)
        for k in range(4):
            out[3, k] += (heat * phi[k] * mesh["vw"]).sum(0)
        for f, pair in zip(mesh["faces"], lifts):
            if pair is None:
                continue
            n, a = f["n"], f["axis"]
            ft, fu, fq = [0.0] * 3, 0.0, 0.0
            for e, b, lift in ((f["e0"], f["b0"], pair[0]), (f["e1"], f["b1"], pair[1])):
                t = _trace(aux[:, :, e] if not self.eta else own[:, :, e] + self.eta * lift, None, b)
                v = self.gas.prim(_trace(x, e, b))["v"]
                mat = [[t[0], t[3], t[4]], [t[3], t[1], t[5]], [t[4], t[5], t[2]]]
                for j in range(3):
                    ft[j] = ft[j] + 0.5 * mat[j][a] * n[a]
                    fu = fu + 0.5 * v[j] * mat[a][j] * n[a]
                fq = fq + 0.5 * t[6 + a] * n[a]
            q = ft + [fu - fq]
            out[:4] -= torch.zeros_like(out[:4]).index_add(2, f["e0"], _moments(q, f["b0"], f["w"]))
            out[:4] += torch.zeros_like(out[:4]).index_add(2, f["e1"], _moments(q, f["b1"], f["w"]))
        return x, out


def _gm_dt(u0, dh):
    rho, ru, re = u0[:, 4, 0], u0[:, 0:3, 0], u0[:, 3, 0]
    p = 0.4 * (re - 0.5 * (ru ** 2).sum(1) / rho)
    return 0.3 * dh / np.sqrt(1.4 * p / rho).max()


def _objective(mesh, gas, u, dt):
    c = (mesh["x"].to(torch.float64) / 1024.0).T + 0.5 * mesh["h"]
    lo, hi = (torch.tensor(b, dtype=torch.float64, device=u.device)[:, None] for b in _PULSE_BOX)
    inside = ((c >= lo) & (c <= hi)).all(0)
    p = gas.prim(_trace(u, None, mesh["vb"]))["p"]
    return dt * ((p * mesh["vw"]).sum(0) * inside).sum()


def exact(case, seed):
    kind = case["kind"]
    if kind == "flux":
        gas = _Gas(**_AIR)
        rows = _flux_rows(case, seed)
        sides = []
        for r in rows[:2]:
            u = np.concatenate([_cons(r[:, 0], r[:, 1:4], r[:, 4])], 1).T
            sides.append(gas.prim(_t(u)))
        return torch.stack(_flux(case["flux"], *sides, _t(rows[2].T))).T.contiguous().cpu().numpy()
    if kind == "multi_tree":
        mesh = _gm_mesh(case["trees"], case["level"])
        c, dh = _gm_centres(case)
        u0 = _flow_state(case, seed, None, c)
        u, dt, gas = _to(u0), _gm_dt(u0, dh), _Gas(**_AIR)
        for _ in range(case["steps"]):
            u = _step(mesh, gas, case["flux"], None, case["limiter"], u, dt)
        return _from(u)
    leaves = _leaves(case)
    mesh = _octree(leaves, case.get("flow") == "sine")
    gas = _Gas(**_gas(case))
    if kind == "steps":
        u0 = _flow_state(case, seed, leaves)
        u = _to(u0)
        s = gas.prim(u[:, 0])
        dt = float((case.get("cfl", 0.3) * mesh["h"] / (torch.sqrt(sum(v * v for v in s["v"])) + s["cz"])).min())
        for _ in range(case["steps"]):
            u = _step(mesh, gas, case["flux"], None, case["limiter"], u, dt)
        return dict(dt=dt, sums=(u[:, 0] * mesh["vol"]).sum(1).cpu().numpy(), state=_from(u))
    if kind == "hot_spot":
        gas = _Gas(W.C4_M, _species())
        dt = _HOT_DT / (1 << case["level"])
        src = _HotSpot(mesh, gas, case["br2_eta"], dt)
        u = _to(_hot_spot_state(leaves, seed))
        for _ in range(case["steps"]):
            u = _step(mesh, gas, "HLLC", None, False, u, dt, source=src)
        return _from(u)
    bc = [_INLET] + [None] * 5
    if kind == "stage_vjp":
        dt = 0.1 / (1 << (case["level"] + case["depth"])) / 1.7
        u0 = _smooth_state(leaves, seed)
        u = _to(u0).requires_grad_()
        x = _to(np.random.default_rng(seed + 1).normal(size=u0.shape))
        y = u - dt * _solve(mesh, _residual(mesh, gas, case["flux"], bc, u))
        return _from(torch.autograd.grad(y, u, x)[0])
    if kind == "adjoint":
        return _exact_adjoint(case, seed, mesh, gas, leaves, bc)
    # the estimator: Green-Gauss density gradient over the faces
    u = _to(_flow_state(dict(case, flow="bubble"), seed, leaves))
    rho = u[4:].sum(0, keepdim=True)
    g = torch.zeros(3, mesh["n"], dtype=u.dtype, device=u.device)
    for f in mesh["faces"]:
        r0 = _trace(rho, f["e0"], f["b0"])[0]
        r1 = r0 if f["e1"] is None else _trace(rho, f["e1"], f["b1"])[0]
        m = (0.5 * (r0 + r1) * f["w"]).sum(0) * f["n"][f["axis"], 0, 0]
        g[f["axis"]].index_add_(0, f["e0"], m)
        if f["e1"] is not None:
            g[f["axis"]].index_add_(0, f["e1"], -m)
    g = g / mesh["vol"]
    return dict(err2=((g * g).sum(0) / 12 * mesh["vol"] ** (5 / 3)).cpu().numpy(), rho=rho[0, 0].cpu().numpy(),
                leaves=None, state=None)


def _exact_adjoint(case, seed, mesh, gas, leaves, bc):
    """reverse mode step by step over stored step states"""
    dt, steps = 0.1 / (1 << case["level"]) / 1.7, case["steps"]
    theta = torch.tensor([_INLET[0], _INLET[3], _INLET[4]], dtype=torch.float64, device=_dev(), requires_grad=True)
    us = [_to(_pulse_state(leaves, seed))]

    def step(u):
        b = [(theta[0], 0.0, 0.0, theta[1], theta[2])] + [None] * 5
        return _step(mesh, gas, "HLLC", b, False, u, dt)
    j = 0.0
    with torch.no_grad():
        for _ in range(steps):
            us.append(step(us[-1]))
            j += float(_objective(mesh, gas, us[-1], dt))
    lam, th = torch.zeros_like(us[0]), torch.zeros(3, dtype=torch.float64, device=_dev())
    for k in range(steps - 1, -1, -1):
        u = us[k].detach().requires_grad_()
        y = step(u)
        out = (y * lam).sum() + _objective(mesh, gas, y, dt)
        lam, dth = torch.autograd.grad(out, (u, theta))
        th = th + dth
    return dict(j=j, grad=_from(lam), theta=th.cpu().numpy())
