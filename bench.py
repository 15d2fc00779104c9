"""Benchmark of the DG residual / time-step path on one MI355X.

Workload: the Riemann-box configuration (Euler P1, uniform octree level 7 =
128^3 = 2,097,152 hexes, HLLC flux + Barth-Jespersen limiter, SSP-RK3,
transmissive boundaries, dt = 0.3 h / max(|u| + c) fixed at t = 0).  Both the
FP32-bulk and the FP64 plain paths run K steps from the same initial state;
value = DOF-updates/s of the FP32 path (E * 4 * V * 3 stages * K / wall).

    python bench.py [--steps K] [--warmup W] [--level L] [--no-fp64] [--no-cpu] [--no-extra]
                    [--no-traffic]

The JSON line also carries the other configurations at full size (adaptive
bubbles, reacting hot spot, adjoint of the pulse case with its FP64 reference
gradient checked against central differences, the Riemann box on a multi-tree
mesh of distorted hexahedra) under "workloads",
the FP32 errors of the smooth cases, the FP64 path's own sensitivity to the
FP32 rounding of the initial state, and the stage kernel's HBM traffic per
launch from two rocprofv3 counter passes (child processes).
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "DOF-updates/s, FP32-mix vs FP64 at L2≤1e-6; %HBM roofline; adjoint/fwd"
HBM_PEAK_GBS = 8000.0
L2_GATE = 1e-6          # the metric's gate on the relative L2 error against the FP64 path


def stage_kernel_bytes(nv, real_bytes):
    """Algorithmic HBM bytes per element of one stage-kernel launch: read the
    stage state and write the new state (4V coefficients each), six int32
    neighbour indices and four geometry words."""
    return real_bytes * 4 * nv * 2 + 4 * 6 + 4 * 4


def step_bytes(nv, real_bytes):
    """Algorithmic bytes per element and RK stage of a whole step: state read
    and write, the extra U^n read of stages 2-3 (2/3 on average), indices and
    geometry: 4 (4V)(2 + 2/3) + 24 + 16 for FP32."""
    return real_bytes * 4 * nv * (2 + 2.0 / 3.0) + 4 * 6 + 4 * 4


def run_path(CA, W, level, precision, steps, warmup, u0=None):
    cfg, leaves, uic, periodic = W.c2(level=level, precision=precision)
    if u0 is None:
        u0 = uic
    ctx = CA.GpuContext(cfg)
    ce, cf = CA.recommended_chunks(cfg)
    if os.environ.get("CHARM_CHUNKS"):
        ce, cf = (int(x) for x in os.environ["CHARM_CHUNKS"].split(","))
    mesh = CA.Forest.from_leaves(leaves, periodic).flatten(ce, cf)
    ctx.upload_mesh(mesh)
    chunking = {"chunk_elems": ce, "chunk_faces": cf, "chunks": mesh.num_chunks, "faces": mesh.num_faces,
                "face_copies_per_face": mesh.num_chunk_faces / mesh.num_faces}
    ctx.set_state(u0)
    dt = ctx.get_dt(mode=1)
    m0 = ctx.conservation_sums()
    if warmup:
        ctx.run(dt, warmup)
        ctx.set_state(u0)
    ctx.synchronize()
    t0 = time.perf_counter()
    ctx.run(dt, steps)
    wall = time.perf_counter() - t0
    dev_ms = ctx.last_ms()
    state = ctx.get_state()
    m1 = ctx.conservation_sums()
    return dict(ctx=ctx, cfg=cfg, leaves=leaves, u0=u0, dt=dt, wall=wall, dev_ms=dev_ms,
                state=state, m0=m0, m1=m1, chunking=chunking)


def cpu_run(W, level, steps, warmup):
    """Child of the CPU baseline (never touches the GPU): the FP64 oracle
    build named by CHARM_ORACLE_LIB on the Riemann box at `level`, `warmup`
    untimed steps, then `steps` timed ones; returns its record."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as OL
    import charm_3d_amd as CA
    cfg, leaves, u0, _ = W.c2(level=level, precision=CA.FP64)
    ocfg = OL.make_config(flux="HLLC", limiter=True, model="NS", bnd=("OUTLET",) * 6)
    t0 = time.perf_counter()
    sim = OL.OracleSim(ocfg, leaves)
    sim.set_state(u0)
    setup = time.perf_counter() - t0
    dt = sim.cfl_dt(1)
    if warmup:
        sim.run(dt, warmup)
    t0 = time.perf_counter()
    sim.run(dt, steps)
    t = time.perf_counter() - t0
    return {"dofs": W.dof_updates(len(leaves), 5, 3, steps), "seconds": t, "steps": steps, "level": level,
            "elements": len(leaves), "setup_s": setup, "lib": os.path.basename(OL.LIB_PATH),
            "threads": int(os.environ.get("OMP_NUM_THREADS", "1"))}


def host_info():
    """lscpu's model name, sockets, cores per socket and logical CPUs"""
    import subprocess
    info = {}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=30).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            info[k.strip()] = v.strip()
    except (OSError, subprocess.SubprocessError):
        pass
    sockets = int(info.get("Socket(s)", "0") or 0)
    cores = int(info.get("Core(s) per socket", "0") or 0)
    return {"model": info.get("Model name", "?"), "physical_cores": sockets * cores or None,
            "logical_cpus": int(info.get("CPU(s)", "0") or 0) or os.cpu_count(),
            "threads_per_core": info.get("Thread(s) per core")}


def cpu_baseline(W, level, threads):
    """The FP64 oracle (the C restatement of the reference numerics: array-
    of-structs leaf records, per-basis field recomputation, callback face
    traversal) on the benchmark's own Riemann box, in child processes that
    never touch the GPU.  The headline is the OpenMP build (leaf- and
    face-parallel passes with the serial sums) at the benchmark's level on
    `threads` threads, 1 warm-up and 3 timed steps; beside it the same build
    on one thread at level 5, and the reference-faithful build (per-leaf
    records and field loops sized for the reference's 128 species, about its
    24 KB per leaf) at level 5 on all threads.  The reference itself needs
    p4est, libsc and yaml-cpp, which are absent, so it cannot be built."""
    import subprocess

    def child(lib, lvl, nthr, steps, warmup):
        env = dict(os.environ, CHARM_ORACLE_LIB=os.path.join(ROOT, "oracle", lib), OMP_NUM_THREADS=str(nthr))
        cmd = [sys.executable, os.path.abspath(__file__), "--cpu-run", str(lvl), str(steps), str(warmup)]
        r = subprocess.run(cmd, env=env, capture_output=True, text=True, timeout=1800)
        if r.returncode != 0:
            return {"error": r.stderr[-400:]}
        rec = json.loads(r.stdout.strip().splitlines()[-1])
        rec["value"] = rec["dofs"] / rec["seconds"]
        return rec

    print("[bench] CPU baseline: level %d, %d threads" % (level, threads), file=sys.stderr, flush=True)
    main_run = child("liboracle_omp.so", level, threads, 3, 1)
    print("[bench] CPU baseline: one thread, reference-faithful records", file=sys.stderr, flush=True)
    single = child("liboracle_omp.so", 5, 1, 3, 1)
    faithful = child("liboracle_faithful.so", 5, threads, 2, 1)
    host = host_info()
    out = {"value": main_run.get("value"), "unit": "DOF-updates/s", "cores": threads, "kind": "port",
           "sample": "FP64 oracle (C restatement of the reference numerics: AoS leaf records, per-basis field "
                     "recomputation, callback face traversal), OpenMP build on %d threads, the benchmark's "
                     "Riemann box at level %d (%s hexes), HLLC + BJ, SSP-RK3: 1 warm-up and 3 timed steps "
                     "(%.1f s)" % (threads, level, main_run.get("elements"), main_run.get("seconds", 0.0)),
           "host": host, "run": main_run,
           "single_thread": single,
           "reference_faithful": dict(faithful, note="per-leaf records and field loops for the reference's "
                                                     "128 species (include/charm_def.h:181), level 5")}
    return out


def rel_errors(a, ref):
    d = a - ref
    return {"l2_rel": float(np.linalg.norm(d) / np.linalg.norm(ref)),
            "linf_rel": float(np.abs(d).max() / np.abs(ref).max()),
            "l2_rel_means": float(np.linalg.norm(d[:, :, 0]) / np.linalg.norm(ref[:, :, 0]))}


def long_run_errors(CA, W, level, u0, steps):
    """The same comparison over `steps` steps (the configuration's 200):
    FP32 and mixed against FP64, and the FP64 path from the FP32-rounded
    initial state (the case's own sensitivity at that length)."""
    print("[bench] %d-step comparison" % steps, file=sys.stderr, flush=True)
    res = {}
    for key, prec, init in (("f64", CA.FP64, u0), ("f32", CA.FP32, u0), ("f32_mix", CA.FP32_MIX, u0),
                            ("f64_rounded", CA.FP64, u0.astype(np.float32).astype(np.float64))):
        r = run_path(CA, W, level, prec, steps, 0, u0=init)
        res[key] = r["state"]
        r["ctx"].close()
    out = {"steps": steps}
    for key in ("f32", "f32_mix"):
        out[key] = rel_errors(res[key], res["f64"])
    out["fp64_from_fp32_rounded_input"] = rel_errors(res["f64_rounded"], res["f64"])
    return out


def smooth_errors(CA, W):
    """FP32 bulk and FP32 mixed (FP64 state, FP32 residual) against the
    FP64 plain path on the two smooth configurations: the advected sine
    wave (level 4, LF, periodic, 100 steps) and the Gaussian pulse (level 6,
    HLLC, inlet, 400 steps); and the FP64 path from the FP32-rounded initial
    state, the case's own sensitivity to a 6e-8 change."""
    out = {}
    cases = (("sine_wave_level4_lf_100_steps", lambda prec: W.c1(4, prec), 100),
             ("gaussian_pulse_level6_hllc_400_steps", lambda prec: W.c5_pulse(6, prec), 400))
    for name, mk, steps in cases:
        res = {}
        for prec in (CA.FP64, CA.FP32, CA.FP32_MIX, "rounded"):
            cfg, leaves, u0, per = mk(CA.FP64 if prec == "rounded" else prec)
            if prec == "rounded":
                u0 = u0.astype(np.float32).astype(np.float64)
            ctx = CA.GpuContext(cfg)
            ce, cf = CA.recommended_chunks(cfg)
            ctx.upload_mesh(CA.Forest.from_leaves(leaves, per).flatten(ce, cf))
            ctx.set_state(u0)
            dt = ctx.get_dt(1) if prec == CA.FP64 else res["dt"]
            m0 = ctx.conservation_sums()
            ctx.run(dt, steps)
            m1 = ctx.conservation_sums()
            res[prec] = ctx.get_state()
            res["dt"] = dt
            res["drift%s" % prec] = abs(m1[4] - m0[4]) / abs(m0[4])
            ctx.close()
        e = rel_errors(res[CA.FP32], res[CA.FP64])
        e["mass_drift_fp32"] = res["drift%s" % CA.FP32]
        e["mass_drift_fp64"] = res["drift%s" % CA.FP64]
        e["fp32_mix"] = rel_errors(res[CA.FP32_MIX], res[CA.FP64])
        e["fp32_mix"]["mass_drift"] = res["drift%s" % CA.FP32_MIX]
        e["fp64_from_fp32_rounded_input"] = rel_errors(res["rounded"], res[CA.FP64])
        out[name] = e
    return out


def traffic_probe(CA, W, level, precision):
    """Child of the traffic measurement: a few stage-kernel and copy-kernel
    launches on the benchmark configuration, nothing else."""
    cfg, leaves, u0, per = W.c2(level=level, precision=precision)
    ctx = CA.GpuContext(cfg)
    ce, cf = CA.recommended_chunks(cfg)
    ctx.upload_mesh(CA.Forest.from_leaves(leaves, per).flatten(ce, cf))
    ctx.set_state(u0)
    dt = ctx.get_dt(mode=1)
    ctx.time_kernels(dt, 3)
    ctx.time_copy(3)
    ctx.synchronize()


def measure_traffic(level, copy_bytes, precision):
    """HBM bytes per stage-kernel launch from two rocprofv3 counter passes
    (FETCH_SIZE, then WRITE_SIZE, KiB per dispatch), each a child process
    running traffic_probe; each counter is scaled by what it reads for the
    copy kernel of known size (copy_bytes / 2 read, copy_bytes / 2 written).
    A third pass reads the stage kernel's VALU instruction counts and busy
    cycles: valu_busy = the issue cycles of its wave64 VALU instructions (4
    each on a 16-lane SIMD, over 4 SIMDs x 256 CUs) over the GPU's busy
    cycles per XCD (GRBM_GUI_ACTIVE summed over the 8 XCDs); the
    quarter-rate transcendentals are counted apart.
    Returns None when rocprofv3 is absent or a pass fails."""
    import csv
    import shutil
    import subprocess
    import tempfile
    prof = shutil.which("rocprofv3")
    if not prof:
        return None
    res = {}
    passes = (("FETCH_SIZE",), ("WRITE_SIZE",), ("SQ_INSTS_VALU", "SQ_INSTS_VALU_TRANS_F32", "GRBM_GUI_ACTIVE"))
    with tempfile.TemporaryDirectory() as tmp:
        for i, ctrs in enumerate(passes):
            d = os.path.join(tmp, "pass%d" % i)
            cmd = [prof, "--pmc", *ctrs, "--output-format", "csv", "-d", d, "-o", "p", "--",
                   sys.executable, os.path.abspath(__file__), "--traffic-probe", "--level", str(level),
                   "--probe-precision", str(precision)]
            print("[bench] counter pass %s" % " ".join(ctrs), file=sys.stderr, flush=True)
            try:
                r = subprocess.run(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=120)
            except subprocess.TimeoutExpired:
                return None
            path = os.path.join(d, "p_counter_collection.csv")
            if r.returncode != 0 or not os.path.exists(path):
                return None
            vals = {}
            for row in csv.DictReader(open(path)):
                k = "stage" if "k_stage" in row["Kernel_Name"] else ("copy" if "k_copy16" in row["Kernel_Name"] else None)
                if k and row["Counter_Name"] in ctrs:
                    vals.setdefault((k, row["Counter_Name"]), []).append(float(row["Counter_Value"]))
            for c in ctrs:
                for k in ("stage", "copy"):
                    v = vals.get((k, c))
                    if not v:
                        return None
                    res[(k, c)] = sum(v) / len(v)
    half = copy_bytes / 2.0
    f_read = half / (res[("copy", "FETCH_SIZE")] * 1024.0)
    f_write = half / (res[("copy", "WRITE_SIZE")] * 1024.0)
    simd_cycles = res[("stage", "SQ_INSTS_VALU")] * 4.0 / 1024.0
    return {"read": res[("stage", "FETCH_SIZE")] * 1024.0 * f_read,
            "write": res[("stage", "WRITE_SIZE")] * 1024.0 * f_write,
            "fetch_scale": f_read, "write_scale": f_write,
            "valu_insts": res[("stage", "SQ_INSTS_VALU")],
            "valu_trans_insts": res[("stage", "SQ_INSTS_VALU_TRANS_F32")],
            "valu_busy": simd_cycles / (res[("stage", "GRBM_GUI_ACTIVE")] / 8.0)}


def extra_workloads(CA, W):
    """The other configurations at their full sizes (FP32), each a few
    seconds: the adaptive bubble case, the reacting hot spot, the adjoint of
    the pulse case (adjoint / forward wall-time ratio) and the Riemann box on
    a multi-tree mesh of distorted hexahedra.  A case
    that fails reports its error instead of a measurement."""
    out = {}
    for name, fn in (("bubbles_adaptive", bench_bubbles), ("reacting_hot_spot", bench_hot_spot),
                     ("pulse_adjoint", bench_adjoint), ("multi_tree_riemann_box", bench_multi_tree)):
        print("[bench]   %s" % name, file=sys.stderr, flush=True)
        try:
            out[name] = fn(CA, W)
        except CA.CharmError as e:
            out[name] = {"error": str(e)}
    return out


def common_leaf_errors(leaves_a, ua, leaves_b, ub):
    """Errors of ua against ub over the leaves both leaf sets hold (two runs
    whose re-adaptations may part ways); the share of common leaves."""
    key_b = {tuple(q): i for i, q in enumerate(np.asarray(leaves_b).tolist())}
    ia, ib = [], []
    for i, q in enumerate(np.asarray(leaves_a).tolist()):
        j = key_b.get(tuple(q))
        if j is not None:
            ia.append(i)
            ib.append(j)
    e = rel_errors(ua[ia], ub[ib])
    e["common_leaf_share"] = len(ia) / max(len(leaves_a), len(leaves_b))
    return e


def bench_bubbles(CA, W):
    # bubbles: levels 5-8 (about 1M leaves), exact Riemann, two species,
    # re-adaptation every 20 steps; FP32 bulk (mixture EOS closure in FP64),
    # then the FP64 path from the same leaves and state for its errors
    t0 = time.perf_counter()
    cfg, forest, u0 = W.c3(precision=CA.FP32)
    t_init = time.perf_counter() - t0
    leaves0 = forest.leaves()
    runs = {}
    for prec in (CA.FP32, CA.FP64):
        if prec == CA.FP64:
            cfg = W.c3_config(CA.FP64, cfg.max_err, cfg.min_level, cfg.max_level)
            forest = CA.Forest.from_leaves(leaves0)
        s = CA.Solver(forest, cfg)
        s.set_state(u0)
        dt = s.get_dt(1) if prec == CA.FP32 else runs[CA.FP32]["dt"]
        m0 = s.conservation_sums()
        gpu_ms, adapt_s, dofs = 0.0, 0.0, 0
        for blk in range(10):
            if blk:
                t = time.perf_counter()
                s.adapt()
                adapt_s += time.perf_counter() - t
            dofs += W.dof_updates(forest.n, 6, 3, 20)
            s.run(dt, 20)
            gpu_ms += s.last_ms()
        m1 = s.conservation_sums()
        runs[prec] = dict(dt=dt, gpu_ms=gpu_ms, adapt_s=adapt_s, dofs=dofs, m0=m0, m1=m1,
                          leaves=forest.leaves(), state=s.get_state(), n=forest.n)
        s.close()
    r = runs[CA.FP32]
    out = {
        "leaves_initial": len(leaves0), "leaves_final": r["n"], "steps": 200, "adapt_every": 20,
        "dof_updates_per_s_device": r["dofs"] / (r["gpu_ms"] * 1e-3),
        "dof_updates_per_s_with_adaptation": r["dofs"] / (r["gpu_ms"] * 1e-3 + r["adapt_s"]),
        "ms_per_step": r["gpu_ms"] / 200, "host_s_per_adaptation": r["adapt_s"] / 9, "init_s": t_init,
        "species_mass_change": [float((r["m1"][4 + i] - r["m0"][4 + i]) / r["m0"][4 + i]) for i in range(2)],
        "eos": "mixture closure (cp, M, gamma) in FP64 arithmetic on the FP32 path"}
    q = runs[CA.FP64]
    mass = lambda m: m[4] + m[5]
    out["fp64"] = {"ms_per_step": q["gpu_ms"] / 200, "leaves_final": q["n"],
                   "species_mass_change": [float((q["m1"][4 + i] - q["m0"][4 + i]) / q["m0"][4 + i]) for i in range(2)]}
    out["errors_vs_fp64"] = common_leaf_errors(r["leaves"], r["state"], q["leaves"], q["state"])
    # conserved mass: the FP32 run's total against the FP64 run's (both lose
    # mass through the transmissive faces alike)
    out["errors_vs_fp64"]["mass_drift"] = float(abs(mass(r["m1"]) - mass(q["m1"])) / abs(mass(q["m0"])))
    return out


def bench_hot_spot(CA, W):
    # reacting hot spot: level 6, four species, BR2 viscous terms, diffusion,
    # chemistry (A = 1e9, molar energy source), 100 steps; FP32 transport with
    # the FP64 Newton temperature and chemistry, then the FP64 path for its
    # errors, then the FP32 path with the reference's BR1 viscous flux
    runs = {}
    for prec, eta in ((CA.FP32, W.C4_BR2_ETA), (CA.FP64, W.C4_BR2_ETA), ("br1", 0.0)):
        cfg, leaves, u0, per = W.c4(6, CA.FP32 if prec == "br1" else prec, visc_br2_eta=eta)
        ctx = CA.GpuContext(cfg)
        ce, cf = CA.recommended_chunks(cfg)
        ctx.upload_mesh(CA.Forest.uniform(6).flatten(ce, cf))
        ctx.set_state(u0)
        dt = ctx.get_dt(1) if prec == CA.FP32 else runs[CA.FP32]["dt"]
        ctx.run(dt, 2)
        ctx.set_state(u0)
        m0 = ctx.conservation_sums()
        ctx.run(dt, 100)
        ms = ctx.last_ms()
        runs[prec] = dict(dt=dt, ms=ms, m0=m0, m1=ctx.conservation_sums(), state=ctx.get_state(), u0=u0)
        ctx.close()
    r, q, b = runs[CA.FP32], runs[CA.FP64], runs["br1"]
    mass = lambda m: m[4:].sum()
    h2o = q["state"][:, 6, 0]
    out = {"leaves": len(leaves), "steps": 100, "ms_per_step": r["ms"] / 100,
           "dof_updates_per_s": W.dof_updates(len(leaves), 8, 3, 100) / (r["ms"] * 1e-3),
           "reaction": "2 H2 + O2 -> 2 H2O, k = A exp(-15000 K / T), A = %g; energy source sum_i w_i M_i h_i "
                       "(the reference's sum_i w_i h_i mixes mol and kg units and fails within two steps "
                       "at this A)" % cfg.react[0].a,
           "viscous_flux": "BR2, eta = %g (the reference's is BR1)" % W.C4_BR2_ETA,
           "br1": {"ms_per_step": b["ms"] / 100, "l2_rel_vs_br2": rel_errors(b["state"], r["state"])["l2_rel"]},
           "fp64": {"ms_per_step": q["ms"] / 100,
                    "mass_drift": float(abs(mass(q["m1"]) - mass(q["m0"])) / mass(q["m0"])),
                    "h2o_mass_max": float(h2o.max() / q["state"][:, 4:, 0].sum(1)[np.argmax(h2o)])},
           "mass_drift": float(abs(mass(r["m1"]) - mass(r["m0"])) / mass(r["m0"])),
           "errors_vs_fp64": rel_errors(r["state"], q["state"])}
    return out


def gmesh_stage_bytes(nv, real_bytes, faces_per_leaf):
    """HBM bytes per leaf of one multi-tree stage (face pass + element pass)
    by design: per face the 33 basis / weight words, the FP64 normal, two
    leaf indices, both sides' states and the face sums written; per leaf its
    54 geometry words (51 and the 3 basis means), the state read and written,
    its six face indices and face sums, 3 basis words of each face where it is
    side 0 and 6 where it is side 1, and its cell means for the limiter."""
    s = real_bytes * 4 * nv
    face = real_bytes * 33 + 8 * 3 + 4 * 2 + 3 * s
    leaf = real_bytes * 54 + 2 * s + 6 * (s + 4) + (faces_per_leaf * 3 + (6 - faces_per_leaf) * 6) * real_bytes + real_bytes * nv
    return faces_per_leaf * face + leaf


def bench_multi_tree(CA, W, steps=20):
    # the Riemann box on 4^3 distorted trees at level 5 (2,097,152 non-affine
    # hexahedra, the octree benchmark's size): FP32 and FP64, 20 steps
    t0 = time.perf_counter()
    runs = {}
    for prec in (CA.FP32, CA.FP64):
        cfg, gm, u0, dt = W.c2_multi_tree(precision=prec)
        t_build = time.perf_counter() - t0
        ctx = CA.GpuContext(cfg)
        ctx.upload_gmesh(gm)
        ctx.set_state(u0)
        ctx.run(dt, 2)
        ctx.set_state(u0)
        ctx.synchronize()
        t = time.perf_counter()
        ctx.run(dt, steps)
        wall = time.perf_counter() - t
        ms = ctx.last_ms()
        state = ctx.get_state()
        ctx.set_state(u0)
        stage_ms, lim_ms = ctx.time_kernels(dt, 10)
        runs[prec] = dict(wall=wall, ms=ms, state=state, stage_ms=stage_ms, lim_ms=lim_ms, n=gm.n, nf=gm.nf,
                          build_s=t_build)
        ctx.close()
        gm.close()
        t0 = time.perf_counter()
    r, q = runs[CA.FP32], runs[CA.FP64]
    n, fpl = r["n"], r["nf"] / r["n"]
    out = {"leaves": n, "faces": r["nf"], "trees": 64, "level": 5, "steps": steps,
           "mesh": "unit box of 4^3 trees, vertices displaced by up to 0.1 of the tree size, refined to level 5",
           "host_mesh_build_s": r["build_s"]}
    for name, x, rb in (("fp32", r, 4), ("fp64", q, 8)):
        b = gmesh_stage_bytes(5, rb, fpl)
        out[name] = {"dof_updates_per_s": W.dof_updates(n, 5, 3, steps) / x["wall"],
                     "ms_per_step": 1e3 * x["wall"] / steps, "device_ms_per_step": x["ms"] / steps,
                     "stage_ms": x["stage_ms"], "limiter_ms": x["lim_ms"], "stage_bytes_per_leaf": b,
                     "stage_hbm_frac": b * n / (x["stage_ms"] * 1e-3) / 1e9 / HBM_PEAK_GBS}
    out["fp32"]["errors_vs_fp64"] = rel_errors(r["state"], q["state"])
    return out


def bench_adjoint(CA, W, fd_check=True):
    # adjoint of the pulse case: level 6, 400 steps, checkpoints every 20
    cfg, leaves, u0, per = W.c5_pulse(6, CA.FP32)
    ctx = CA.GpuContext(cfg)
    ce, cf = CA.recommended_chunks(cfg)
    ctx.upload_mesh(CA.Forest.uniform(6).flatten(ce, cf))
    ctx.set_state(u0)
    dt = ctx.get_dt(1)
    lo, hi = W.C5_BOX
    J, g, th, fwd_ms, adj_ms = ctx.adjoint(dt, 400, lo, hi, ckpt=20, theta_face=0)
    # the memory-rich variant: every stage state of the forward pass kept
    # (1,201 states, 25 GB at this size), no recompute; the same gradient
    ctx.set_state(u0)
    J0, g0, th0, fwd0, adj0 = ctx.adjoint(dt, 400, lo, hi, ckpt=0, theta_face=0)
    ctx.close()
    out = {"leaves": len(leaves), "steps": 400, "checkpoint_every": 20, "J": J,
           "dJ_dinlet_u_T_p": th.tolist(), "forward_ms": fwd_ms, "adjoint_ms": adj_ms,
           "adjoint_over_forward": adj_ms / fwd_ms,
           "all_stage_states_kept": {"forward_ms": fwd0, "adjoint_ms": adj0, "adjoint_over_forward": adj0 / fwd0,
                                     "same_gradient_bits": bool(J0 == J and np.array_equal(g0, g)
                                                                and np.array_equal(th0, th))}}
    if fd_check:
        out["fp64_reference"] = adjoint_fd_check(CA, W, dt, g, th)
    return out


def adjoint_fd_check(CA, W, dt, g32, th32, ndir=32, steps=(1e-6, 1e-7)):
    """The FP64 adjoint of the same case, checked against central differences
    of the FP64 forward objective: dJ/du0 along ndir random directions
    (per-variable scaled), dJ/d(inlet u, T, p) per parameter, each at the
    relative steps in `steps`; and the FP32 gradient against the FP64 one.
    The objective has kinks (the switch of the HLLC wave-speed factor at
    p* = p_k, min / max of the wave speeds), so a central difference carries an
    error linear in h wherever a perturbation moves a face point across one;
    the adjoint is the derivative of the branch taken."""
    lo, hi = W.C5_BOX
    inlet = np.array([0.5, 1.0, 1.0])

    def device(u, theta):
        cfg, leaves, u0, per = W.c5_pulse(6, CA.FP64, inlet=tuple(theta))
        ctx = CA.GpuContext(cfg)
        ce, cf = CA.recommended_chunks(cfg)
        ctx.upload_mesh(CA.Forest.uniform(6).flatten(ce, cf))
        ctx.set_state(u0 if u is None else u)
        return ctx, u0

    ctx, u0 = device(None, inlet)
    J, g, th, fwd_ms, adj_ms = ctx.adjoint(dt, 400, lo, hi, ckpt=20, theta_face=0)
    rng = np.random.default_rng(32)
    scale = np.abs(u0).max(axis=0, keepdims=True)
    dirs = [rng.normal(size=u0.shape) * scale for _ in range(ndir)]
    ad = np.array([float((g * v).sum()) for v in dirs])
    cd = {}
    for h in steps:
        fd = []
        for v in dirs:
            ctx.set_state(u0 + h * v)
            jp = ctx.objective(dt, 400, lo, hi)
            ctx.set_state(u0 - h * v)
            jm = ctx.objective(dt, 400, lo, hi)
            fd.append((jp - jm) / (2 * h))
        fd = np.array(fd)
        rel = np.abs(ad - fd) / np.abs(fd)
        worst_th = 0.0
        for k in range(3):
            step = h * max(abs(inlet[k]), 1.0)
            jj = []
            for sgn in (1, -1):
                t = inlet.copy()
                t[k] += sgn * step
                c, _ = device(u0, t)
                jj.append(c.objective(dt, 400, lo, hi))
                c.close()
            fdt = (jj[0] - jj[1]) / (2 * step)
            worst_th = max(worst_th, abs(th[k] - fdt) / abs(fdt))
        cd["h=%g" % h] = {"directions": ndir, "worst_rel_diff_du0": float(rel.max()),
                          "median_rel_diff_du0": float(np.median(rel)),
                          "worst_diff_over_rms_du0": float(np.abs(ad - fd).max() / np.sqrt((ad ** 2).mean())),
                          "worst_rel_diff_dinlet": worst_th}
        if h == steps[0]:
            # the kinks behind the worst directions: the face points whose HLLC
            # branch differs between the +h and -h runs, at the start of each
            # of the 400 steps, for the three worst and the three best
            # directions
            order = np.argsort(rel)
            rows = []
            for i in list(order[-3:][::-1]) + list(order[:3]):
                cp, _ = device(u0 + h * dirs[i], inlet)
                cm, _ = device(u0 - h * dirs[i], inlet)
                tot, npts, bits, first = 0, 0, np.zeros(9, dtype=np.int64), None
                for _ in range(400):
                    pts, fl, pb = cp.hllc_branch_flips(cm, per_bit=True)
                    if first is None:
                        first = fl / pts
                    tot += fl
                    npts += pts
                    bits += pb
                    cp.run(dt, 1)
                    cm.run(dt, 1)
                cp.close()
                cm.close()
                rows.append({"rel_diff": float(rel[i]), "flipped_fraction": tot / npts,
                             "flipped_fraction_step0": first,
                             "by_condition": dict(zip(("p*>pL", "p*>pR", "swap", "SL>=0", "SR<=0", "S*>=0",
                                                       "S*=SL", "S*=SR", "pvrs<=0"), (bits / npts).tolist()))})
            cd["h=%g" % h]["hllc_branch_flips_worst3_best3"] = rows
    ctx.close()
    return {"J": J, "dJ_dinlet_u_T_p": th.tolist(), "forward_ms": fwd_ms, "adjoint_ms": adj_ms,
            "central_differences": cd,
            "fp32_gradient_vs_fp64": {"l2_rel_du0": float(np.linalg.norm(g32 - g) / np.linalg.norm(g)),
                                      "max_rel_dinlet": float(np.abs((th32 - th) / th).max())}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--level", type=int, default=7)
    ap.add_argument("--no-long", action="store_true", help="skip the 200-step error comparison")
    ap.add_argument("--long-steps", type=int, default=200)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extra", action="store_true")
    ap.add_argument("--cpu-level", type=int, default=None,
                    help="level of the CPU baseline's Riemann box (default: the benchmark's)")
    ap.add_argument("--cpu-threads", type=int, default=None,
                    help="OpenMP threads of the CPU baseline (default: OMP_NUM_THREADS, else all CPUs)")
    ap.add_argument("--kernel-reps", type=int, default=20)
    ap.add_argument("--no-traffic", action="store_true")
    ap.add_argument("--traffic-probe", action="store_true", help=argparse.SUPPRESS)
    ap.add_argument("--probe-precision", type=int, default=1, help=argparse.SUPPRESS)
    ap.add_argument("--cpu-run", type=int, nargs=3, default=None, help=argparse.SUPPRESS)
    ap.add_argument("--no-fd-check", action="store_true",
                    help="with --only adjoint: the FP32 adjoint and its timing, without the FP64 reference gradient")
    ap.add_argument("--only", choices=("bubbles", "hot_spot", "adjoint", "multi_tree"),
                    help="run one of the other configurations alone and print its JSON")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(run with --gpus 1)", file=sys.stderr)
        sys.exit(2)

    import charm_3d_amd.workloads as W
    if args.cpu_run:
        print(json.dumps(cpu_run(W, *args.cpu_run)))
        return
    import charm_3d_amd as CA

    if args.traffic_probe:
        traffic_probe(CA, W, args.level, args.probe_precision)
        return
    if args.only:
        fn = {"bubbles": bench_bubbles, "hot_spot": bench_hot_spot, "multi_tree": bench_multi_tree,
              "adjoint": lambda CA, W: bench_adjoint(CA, W, fd_check=not args.no_fd_check)}[args.only]
        print(json.dumps(fn(CA, W)))
        return

    print("[bench] FP32 bulk path, level %d, %d steps" % (args.level, args.steps), file=sys.stderr, flush=True)
    r32 = run_path(CA, W, args.level, CA.FP32, args.steps, args.warmup)
    n = len(r32["leaves"])
    nv = 5
    dofs = W.dof_updates(n, nv, 3, args.steps)
    print("[bench] mixed path (FP64 state, FP32 residual)", file=sys.stderr, flush=True)
    rmx = run_path(CA, W, args.level, CA.FP32_MIX, args.steps, args.warmup, u0=r32["u0"])
    print("[bench] FP64 plain path", file=sys.stderr, flush=True)
    r64 = run_path(CA, W, args.level, CA.FP64, args.steps, min(args.warmup, 2), u0=r32["u0"])

    # the headline is the fastest path whose L2 error against the FP64 path
    # meets the metric's gate at this run's step count; FP64 otherwise
    paths = {"f32": r32, "f32_mix": rmx, "f64": r64}
    gate = {"l2_rel_max": L2_GATE, "steps": args.steps}
    for name in ("f32", "f32_mix"):
        e = rel_errors(paths[name]["state"], r64["state"])
        gate[name] = {"l2_rel": e["l2_rel"], "passed": e["l2_rel"] <= L2_GATE}
    passing = [k for k in ("f32", "f32_mix") if gate[k]["passed"]]
    head = min(passing, key=lambda k: paths[k]["wall"]) if passing else "f64"
    rh = paths[head]
    real_bytes = 4 if head == "f32" else 8          # the stage kernel's state words

    # dominant kernel: the headline path's stage kernel, timed with HIP
    # events on its context's stream
    ctx = rh["ctx"]
    ctx.set_state(rh["u0"])
    stage_ms, lim_ms = ctx.time_kernels(rh["dt"], args.kernel_reps)
    copy_ms, copy_bytes = ctx.time_copy(args.kernel_reps)
    kb = stage_kernel_bytes(nv, real_bytes) * n
    achieved = kb / (stage_ms * 1e-3) / 1e9

    out = {
        "metric": METRIC,
        "value": dofs / rh["wall"],
        "unit": "DOF-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * rh["wall"] / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"f32": "f32", "f32_mix": "f32 (f64 state)", "f64": "f64"}[head],
        "data": "synthetic",
        "headline_path": head,
        "gate": gate,
        "gate_passed": head != "f64",
        "config": {"workload": "Riemann box (rho,p)=(1,1)|(0.125,0.1) at x=0.5 with seeded "
                               "+-1%% cell-mean perturbation, Euler P1 Taylor basis, uniform "
                               "octree level %d (%d hexes), HLLC flux + Barth-Jespersen limiter, "
                               "SSP-RK3, transmissive boundaries, dt = 0.3 h / max(|u|+c)" % (args.level, n),
                   "elements": n, "vars": nv, "stages_per_step": 3, "dt": r32["dt"],
                   "chunking": r32["chunking"]},
        "roofline": {"bound": "hbm", "kernel": "k_stage (fused face flux + volume + gather + update), %s path" % head,
                     "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": None,
                     "stage_ms": stage_ms, "limiter_ms": lim_ms,
                     "bytes_per_elem": stage_kernel_bytes(nv, real_bytes),
                     "copy_GBs": copy_bytes / (copy_ms * 1e-3) / 1e9},
        "whole_step": {"device_ms_per_step": rh["dev_ms"] / args.steps,
                       "algorithmic_GBs": step_bytes(nv, real_bytes) * n * 3 * args.steps / rh["wall"] / 1e9,
                       "hbm_frac": step_bytes(nv, real_bytes) * n * 3 * args.steps / rh["wall"] / 1e9 / HBM_PEAK_GBS},
        "adjoint_over_forward": None,
    }
    for name, r in paths.items():
        rec = {"value": dofs / r["wall"], "ms_per_step": 1e3 * r["wall"] / args.steps,
               "mass_drift": abs(r["m1"][4] - r["m0"][4]) / abs(r["m0"][4])}
        if name != "f64":
            rec["errors_vs_fp64"] = rel_errors(r["state"], r64["state"])
        out[{"f32": "fp32", "f32_mix": "fp32_mix", "f64": "fp64"}[name]] = rec
    if head == "f64":
        out["errors_vs_fp64"] = {"l2_rel": 0.0, "linf_rel": 0.0,
                                 "note": "the headline path is the FP64 path (parity with the oracle: 1e-12)"}
    else:
        out["errors_vs_fp64"] = out[{"f32": "fp32", "f32_mix": "fp32_mix"}[head]]["errors_vs_fp64"]
    out["speedup_fp32_over_fp64"] = r64["wall"] / r32["wall"]
    # conditioning of the case: the FP64 path from the initial state rounded
    # to FP32 (the only difference), against the FP64 run
    print("[bench] FP64 path from the FP32-rounded initial state", file=sys.stderr, flush=True)
    u0r = r32["u0"].astype(np.float32).astype(np.float64)
    r64r = run_path(CA, W, args.level, CA.FP64, args.steps, 0, u0=u0r)
    out["fp64_from_fp32_rounded_input"] = rel_errors(r64r["state"], r64["state"])
    r64r["ctx"].close()
    del r64r
    if not args.no_long:
        out["long_run"] = long_run_errors(CA, W, args.level, r32["u0"], args.long_steps)

    # the level-7 contexts are done with: release their memory and HIP
    # streams before the other workloads (the adjoint overlaps two streams,
    # which need hardware queues of their own)
    for r in paths.values():
        r["ctx"].close()
    del paths, r32, rmx, r64, rh

    if not args.no_extra:
        print("[bench] smooth cases, FP32 against FP64", file=sys.stderr, flush=True)
        out["smooth_errors_vs_fp64"] = smooth_errors(CA, W)
        print("[bench] bubble, hot-spot and adjoint cases", file=sys.stderr, flush=True)
        out["workloads"] = extra_workloads(CA, W)
        out["adjoint_over_forward"] = out["workloads"]["pulse_adjoint"].get("adjoint_over_forward")

    if not args.no_traffic:
        prec = {"f32": CA.FP32, "f32_mix": CA.FP32_MIX, "f64": CA.FP64}[head]
        tr = measure_traffic(args.level, copy_bytes, prec)
        if tr:
            out["roofline"]["traffic"] = tr["read"] + tr["write"]
            out["roofline"]["traffic_detail"] = {k: tr[k] for k in ("read", "write", "fetch_scale", "write_scale")}
            # the bound the stage kernel actually sits at: its VALU issue
            # rate (issue cycles of its VALU instructions over its busy
            # cycles: the VALU-roofline fraction beside the HBM one)
            out["roofline"]["valu"] = {k: tr[k] for k in ("valu_insts", "valu_trans_insts", "valu_busy")}
            out["roofline"]["valu_frac"] = tr["valu_busy"]
            out["roofline"]["valu_insts_per_elem"] = tr["valu_insts"] * 64.0 / n
            if tr["valu_busy"] > out["roofline"]["frac"]:
                out["roofline"]["bound"] = "valu"

    if not args.no_cpu:
        threads = args.cpu_threads or int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or os.cpu_count() or 1
        out["cpu_baseline"] = cpu_baseline(W, args.cpu_level or args.level, threads)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
