"""Benchmark: SSP-Knoth Rosenbrock-W steps of the spectral-element dynamical
core on one MI355X, FP64 (cubed sphere ne=60, p=4, nz=64, 34.56 M element
points, dt=50 s, seeded baroclinic-jet state), with the mixed-precision step
of the same workload, the batched ensemble and the adjoint beside it, the
FP64 drop-in at ne=30 (dt=100 s) as a secondary line, and the FP64 step on
one GPU's share of an 8-way horizontal decomposition of the workload.

Prints one JSON line (rank 0): throughput in element points x steps per
second (Mpts/s, points = 6 ne^2 (p+1)^2 nz), the roofline of the dominant
kernel (fused tendency pass, HBM bound) and the CPU oracle timed on this
host as a reported baseline.
"""
from __future__ import annotations

import argparse
import hashlib
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0  # MI355X HBM3E peak, GB/s
PASS2, ALL_PASSES = 2, 7  # cgd_profile_enable masks


def survey_bytes(ne, p, nz, wt=8, wm=8, wc=8, nf=None, num_g=None):
    """Algorithmic HBM bytes (frozen per-unit formulas of the build's survey).

    Returns dict with per-RW-step total and the per-evaluation bytes of the
    pass-1, pass-2 and column kernels for stage 1.  ``nf``, ``num_g``: the
    element and node counts of a part of the grid (default: the whole
    cubed sphere).
    """
    NE = 6 * ne * ne if nf is None else nf
    N = p + 1
    Ne = NE * N * N * nz
    Ng = ((6 * ne * ne * p * p + 2) if num_g is None else num_g) * nz
    glob = NE * N * N * 8
    pass1 = (4 * Ng * wt + 10 * Ne * wm + 2 * Ng * wm + 5 * Ng * wt) + glob
    pass2 = (5 * Ng * wt + 5 * Ng * wt + 26 * Ne * wm + 2 * Ng * wm + 5 * Ng * wt) + glob
    step = 0
    for i in range(1, 4):
        col = 5 * Ng * wc + (i - 1) * 5 * Ng * wc + (8 + 3) * Ng * wc + 5 * Ng * wc
        stage = (5 + (i - 1) * 5 + 5) * Ng * wc if i >= 2 else 0
        step += pass1 + pass2 + col + stage
    step += (2 * Ng + Ng) * wc + 8 * Ng * wc  # Jacobian
    step += 8 * Ng * wc + 3 * Ng * wc  # tri build
    step += (5 + 15 + 5) * Ng * wc  # final update
    return dict(step=step, pass1=pass1, pass2=pass2, Ne=Ne, Ng=Ng)


KERNEL_DIR = os.path.join(ROOT, "cgdycore.jl_amd", "csrc")


def kernel_source_hash():
    """SHA-256 (first 16 hex digits) of the element-kernel source
    (cgd_kernels.hip and the kernel bodies it includes): a profile summary
    measured on other kernels than the ones running is stale."""
    h = hashlib.sha256()
    for name in ["cgd_kernels.hip"] + sorted(f for f in os.listdir(KERNEL_DIR) if f.endswith("_body.inc")):
        with open(os.path.join(KERNEL_DIR, name), "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def measured_traffic(kernel, workload, algorithmic):
    """HBM bytes per tendency evaluation of ``kernel`` from the committed
    rocprofv3 FETCH_SIZE/WRITE_SIZE summary of the same workload (each counter
    scaled by its reading for a plain copy of known size), or None when there
    is none, or when it was measured on another algorithmic byte count or
    another kernel source than the one built here."""
    path = os.path.join(ROOT, "profiles", f"traffic_{kernel}_{workload}.json")
    try:
        with open(path) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    if t.get("algorithmic_bytes_per_eval") != algorithmic:
        return None
    if t.get("kernel_source_sha16") != kernel_source_hash():
        return None
    return t["traffic_bytes_per_eval"]


def trace_average(kernel, workload):
    """The committed rocprofv3 kernel-trace summary of the same workload
    (profiles/kernels_<workload>.json): average duration of ``kernel``'s
    dispatches in microseconds and the kernel source it was measured on."""
    path = os.path.join(ROOT, "profiles", f"kernels_{workload}.json")
    try:
        with open(path) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    for row in t.get("kernels", []):
        if row.get("name", "").startswith(kernel):
            return {"avg_us": row["avg_us"], "calls": row["calls"],
                    "kernel_source_sha16": t.get("kernel_source_sha16"),
                    "current_source": t.get("kernel_source_sha16") == kernel_source_hash()}
    return None


def mixed_precision(host, disc, phys, U0, args, fp64_ms, V_fp64):
    """The same steps from the same initial state with the tendency and DSS
    in FP32 (FP64 EOS, w-interface balance, horizontal pressure gradient and
    column solve): throughput, and relative L2 / Linf error per prognostic
    variable against the FP64 state after the same number of steps."""
    import torch

    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, hyperd=args.hyperd, device="cuda:0",
                                                          precision="mixed")
    ctx = host.init_context(FE, Metric, phys, Global)
    V = torch.as_tensor(U0, device="cuda:0").clone()
    shape = ctx.launch_shape()
    if not args.no_autotune:
        shape, _ = ctx.autotune(V, args.dt, Cache, JCache, reps=3)

    host.TimeStepper(V, args.dt, args.warmup, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    host.TimeStepper(V, args.dt, args.steps, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms = wall / args.steps * 1e3
    names = ("rho", "u", "v", "w", "rhotheta")
    rel_l2, rel_linf = {}, {}
    for c, n in enumerate(names):
        d = (V[c] - V_fp64[c]).double()
        ref = V_fp64[c].double()
        rel_l2[n] = float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(ref))
        rel_linf[n] = float(d.abs().max() / ref.abs().max())
    # per-pass breakdown from a few extra steps with every pass bracketed
    nb = min(args.steps, 5)
    ctx.profile(ALL_PASSES)
    host.TimeStepper(V, args.dt, nb, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    passes = {name: round(ctx.profile_read(i)[0] / nb, 4) for i, name in enumerate(("pass1", "pass2", "column"))}
    ctx.profile(0)
    Global._ctx.close()
    return {"value": round(disc.element_points * args.steps / wall / 1e6, 2), "unit": "Mpts/s",
            "ms_per_step": round(ms, 4), "speedup_vs_fp64": round(fp64_ms / ms, 3),
            "steps_compared": args.warmup + args.steps, "rel_l2_vs_fp64": rel_l2, "rel_linf_vs_fp64": rel_linf,
            "pass_ms_per_step": passes, "launch_shape": shape,
            "precision": "FP32 tendency and DSS; FP64 EOS, w-interface balance, horizontal pressure gradient, "
                         "column solve and stage arithmetic"}


def ensemble(pkg, args):
    """The batched-ensemble workload: args.ens_members members (theta-noise
    seeds 0..n-1) on cubed spheres ne = 8, 12, 16 (member m on
    (8, 12, 16)[m mod 3]), p = 4, nz = 32, dt = args.ens_dt, one batch
    context, launch shapes from the autotuner, the timed steps replayed
    from one captured HIP graph (one launch).  Reports the mixed-precision
    batch, the FP64 batch and the FP64 members stepped one context at a
    time (the sum of the per-grid step times, each grid timed on its own
    context), with the mixed batch's error against the FP64 batch after the
    same steps."""
    import torch

    host = pkg.host
    D = pkg.discretization
    phys = D.Phys()
    nes, seeds = pkg.state.ensemble_members(args.ens_members)
    nz, dt, K, W = 32, args.ens_dt, args.ens_steps, 1
    grids = {ne: D.build(ne, 4, nz, 30000.0) for ne in sorted(set(nes))}
    discs = [grids[ne] for ne in nes]
    U0 = pkg.state.ensemble_state(discs, seeds)
    points = sum(d.element_points for d in discs)

    def timed(fn, nsteps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(nsteps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / nsteps * 1e3

    out = {"members": len(nes), "grids": {str(ne): nes.count(ne) for ne in sorted(set(nes))}, "p": 4, "nz": nz,
           "dt": dt, "steps": K, "points": points}
    finals = {}
    for prec in ("fp64", "mixed"):
        ens = host.ensemble_setup(discs, phys, precision=prec, device="cuda:0")
        ctx = ens.Global._ctx
        V = torch.as_tensor(U0, device="cuda:0").clone()
        shape, tune_ms = ctx.autotune(V, dt, ens.Cache, ens.JCache, reps=3)
        ctx.graph_create(V, dt, ens.Cache, ens.JCache, nsteps=K)
        for _ in range(W):
            ctx.graph_launch()
        ms = timed(ctx.graph_launch, 1) / K
        finals[prec] = V.clone()
        out[prec] = {"value": round(points / ms / 1e3, 2), "unit": "Mpts/s", "ms_per_step": round(ms, 4),
                     "launch_shape": shape,
                     "finite": bool(torch.isfinite(V).all().item())}
        # each stage as one persistent launch (grid barriers between the
        # passes) against separate launches, both replayed from
        # a captured graph with the persistent kernel's shape fields
        cmp = {}
        for pers in (-1, 1):
            ctx.set_launch_shape(chunk_levels=8, pass1_chunk_levels=8, pass1_items=1, col_lanes=shape["col_lanes"],
                                 col_block=256, persistent=pers)
            Vp = torch.as_tensor(U0, device="cuda:0").clone()
            ctx.graph_create(Vp, dt, ens.Cache, ens.JCache, nsteps=K)
            ctx.graph_launch()
            cmp["persistent" if pers == 1 else "separate"] = round(timed(ctx.graph_launch, 1) / K, 4)
            ctx.check_device()
            del Vp
        out[prec]["one_persistent_launch_per_stage_ms"] = cmp["persistent"]
        out[prec]["separate_launches_same_shape_ms"] = cmp["separate"]
        ctx.close()
        del ens, V
        torch.cuda.empty_cache()
    out["mixed"]["speedup_vs_fp64_batch"] = round(out["fp64"]["ms_per_step"] / out["mixed"]["ms_per_step"], 3)
    rel = {}
    for c, n in enumerate(("rho", "u", "v", "w", "rhotheta")):
        d = (finals["mixed"][c] - finals["fp64"][c]).double()
        rel[n] = float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(finals["fp64"][c].double()))
    out["mixed"]["rel_l2_vs_fp64_batch"] = rel
    out["mixed"]["steps_compared"] = (W + 1) * K
    # the same members without batching: one FP64 context per grid, the
    # step time of each member taken from its grid's context
    per_grid = {}
    for ne, disc in grids.items():
        FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda:0")
        host.init_context(FE, Metric, phys, Global)
        V = torch.as_tensor(pkg.state.jet_state(disc, seed=0), device="cuda:0").clone()

        host.TimeStepper(V, dt, 1, FE, Metric, phys, Cache, JCache, Global)
        per_grid[ne] = timed(lambda: host.TimeStepper(V, dt, K, FE, Metric, phys, Cache, JCache, Global), 1) / K
        Global._ctx.close()
    seq_ms = sum(per_grid[ne] for ne in nes)
    out["fp64_one_member_at_a_time"] = {"ms_per_step": round(seq_ms, 4),
                                        "value": round(points / seq_ms / 1e3, 2), "unit": "Mpts/s",
                                        "ms_per_step_per_grid": {str(k): round(v, 4) for k, v in per_grid.items()}}
    out["batch_speedup_fp64"] = round(seq_ms / out["fp64"]["ms_per_step"], 3)
    return out


def adjoint(pkg, args):
    """The adjoint workload: ne = 16, p = 4, nz = 32, FP64, the seeded jet
    (seed 0); functional J = sum over the lowest level's global nodes of
    rho*theta^2 = (rho theta)^2 / rho after 12 steps at dt = 200 s (at
    dt = 250 or 300 s the step itself -- the C oracle's restatement of the
    reference as well as this path -- diverges within 12 steps at ne = 16:
    horizontal acoustics are explicit in this Rosenbrock-W).  The
    gradient dJ/dV0 comes from the forward with a checkpoint every 4 steps
    (cgd_rw_forward_ckpt, which also gives the final state J needs) and the
    reverse sweep from those checkpoints (cgd_rw_adjoint_ckpt); "ms_gradient"
    times both.  It is checked against central differences
    (J(V0 + eps d) - J(V0 - eps d)) / (2 eps), eps = 1e-6, of the fused
    forward (cgd_rw_run) along 64 Gaussian directions d ~ N(0, 1) per state
    entry (numpy generators seeded 1000..1063; w at the model top, which
    the step keeps fixed, is not perturbed).  J is summed exactly (fsum).
    The same is done twice: with the reference's exact upwind flux, whose
    kinks (|wCon|, the RecU4 limiter) finite differences cross, and in the
    kink-smoothed mode (SmoothW = SmoothC = 1e-2), where the forecast is
    differentiable and the 1e-6 bar applies ("smoothed")."""
    out = _adjoint_case(pkg, args, None)
    out["smoothed"] = _adjoint_case(pkg, args, (1e-2, 1e-2))
    return out


def _adjoint_case(pkg, args, smooth):
    import math

    import torch

    host = pkg.host
    D = pkg.discretization
    ne, nz, dt, nsteps, every, ndir, eps = 16, 32, 200.0, 12, 4, args.adj_dirs, 1e-6
    phys = D.Phys()
    disc = D.build(ne, 4, nz, 30000.0)
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda:0", smooth=smooth)
    ctx = host.init_context(FE, Metric, phys, Global)
    U0 = pkg.state.jet_state(disc, seed=0)
    V0 = torch.as_tensor(U0, device="cuda:0")

    def J_of(Vf):
        lev = Vf[:, :, 0].cpu().numpy()
        return math.fsum((lev[4] ** 2 / lev[0]).tolist())

    def run(V):
        Vt = V.clone()
        host.TimeStepper(Vt, dt, nsteps, FE, Metric, phys, Cache, JCache, Global)
        return Vt

    work = ctx.adjoint_work(nsteps, every, device="cuda:0")
    Vf = torch.empty_like(V0)

    def grad():
        # the rrule's forward keeps its checkpoints; the pullback uses them
        ctx.rw_forward_ckpt(V0, dt, nsteps, every, Vf, work)
        lam = torch.zeros_like(V0)
        lam[4, :, 0] = 2.0 * Vf[4, :, 0] / Vf[0, :, 0]
        lam[0, :, 0] = -(Vf[4, :, 0] / Vf[0, :, 0]) ** 2
        ctx.rw_adjoint_ckpt(dt, nsteps, every, lam, work)
        return lam

    grad()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    g = grad()
    torch.cuda.synchronize()
    t_grad = time.perf_counter() - t0
    t0 = time.perf_counter()
    run(V0)
    torch.cuda.synchronize()
    t_fwd = time.perf_counter() - t0
    gn = g.cpu().numpy()
    errs = []
    for seed in range(1000, 1000 + ndir):
        d = np.random.default_rng(seed).standard_normal(U0.shape)
        d[3][:, -1] = 0.0
        dt_ = torch.as_tensor(d, device="cuda:0")
        fd = (J_of(run(V0 + eps * dt_)) - J_of(run(V0 - eps * dt_))) / (2 * eps)
        ad = float(np.vdot(gn, d))
        errs.append(abs(fd - ad) / abs(fd))
    errs = np.array(errs)
    out = {"ne": ne, "p": 4, "nz": nz, "dt": dt, "steps": nsteps, "checkpoint_every": every, "precision": "fp64",
           "functional": "sum over lowest-level global nodes of rho*theta^2 after the steps",
           "flux": "exact (reference)" if smooth is None else f"kink-smoothed (SmoothW, SmoothC) = {list(smooth)}",
           "J": J_of(Vf), "ms_gradient": round(t_grad * 1e3, 3), "ms_forward": round(t_fwd * 1e3, 3),
           "gradient_over_forward": round(t_grad / t_fwd, 2),
           "fd": {"eps": eps, "directions": ndir, "seeds": f"1000..{1000 + ndir - 1}",
                  "max_rel_err": float(errs.max()), "median_rel_err": float(np.median(errs)),
                  "pass_1e-6": bool(errs.max() <= 1e-6)}}
    ctx.close()
    return out


def secondary(pkg, args):
    """The FP64 drop-in workload at ne=30, p=4, nz=64, dt=100 s: 20 steps
    after 2 warm-up steps, on its own context with autotuned launch shapes
    (the same timing as the headline)."""
    import torch

    host = pkg.host
    D = pkg.discretization
    ne, nz, dt, K, W = 30, 64, 100.0, 20, 2
    disc = D.build(ne, args.p, nz, 30000.0)
    phys = D.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda:0")
    ctx = host.init_context(FE, Metric, phys, Global)
    V = torch.as_tensor(pkg.state.jet_state(disc, seed=0), device="cuda:0").clone()
    shape = ctx.launch_shape()
    if not args.no_autotune:
        shape, _ = ctx.autotune(V, dt, Cache, JCache, reps=3)
    host.TimeStepper(V, dt, W, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    host.TimeStepper(V, dt, K, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    sb = survey_bytes(ne, args.p, nz)
    out = {"workload": f"rw_step_fp64_ne{ne}_p{args.p}_nz{nz}", "value": round(sb["Ne"] * K / wall / 1e6, 2),
           "unit": "Mpts/s", "ms_per_step": round(wall / K * 1e3, 4), "dt": dt, "steps": K, "warmup": W,
           "step_roofline_frac": round(sb["step"] / (wall / K) / 1e9 / PEAK_HBM_GBS, 4),
           "finite": bool(torch.isfinite(V).all().item()), "launch_shape": shape}
    ctx.close()
    return out


def rank_share(pkg, args, disc):
    """One GPU's share of the workload in a horizontal domain decomposition
    into args.share_parts parts (discretization.share, part 0: at ne=60 and
    8 parts, 45 rows of 60 elements of the first cube face), FP64, the
    headline's dt, warm-up and step count, on its own context with autotuned
    launch shapes.  After each DSS a multi-GPU run would sum the share's
    boundary nodes with its neighbours' (a halo exchange, left out on one
    GPU); the bytes it would exchange are reported."""
    import torch

    host = pkg.host
    D = pkg.discretization
    parts = args.share_parts
    sd = D.share(disc, parts, 0)
    nbound = int(D.share_boundary_nodes(disc, parts, 0).size)
    phys = D.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(sd, phys, hyperd=args.hyperd, device="cuda:0")
    ctx = host.init_context(FE, Metric, phys, Global)
    V = torch.as_tensor(pkg.state.jet_state(sd, seed=0), device="cuda:0").clone()
    shape = ctx.launch_shape()
    if not args.no_autotune:
        shape, _ = ctx.autotune(V, args.dt, Cache, JCache, reps=3)
    host.TimeStepper(V, args.dt, args.warmup, FE, Metric, phys, Cache, JCache, Global)
    ctx.profile(PASS2)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    host.TimeStepper(V, args.dt, args.steps, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    p2_ms, _ = ctx.profile_read(1)
    ctx.profile(0)
    sb = survey_bytes(args.ne, args.p, args.nz, nf=sd.nf, num_g=sd.num_g)
    p2_eval_s = p2_ms / 1e3 / (3 * args.steps)
    out = {"workload": f"rw_step_fp64_ne{args.ne}_p{args.p}_nz{args.nz}_part0of{parts}", "parts": parts,
           "elements": sd.nf, "num_g": sd.num_g, "points": sb["Ne"],
           "value": round(sb["Ne"] * args.steps / wall / 1e6, 2), "unit": "Mpts/s",
           "ms_per_step": round(wall / args.steps * 1e3, 4), "dt": args.dt, "steps": args.steps,
           "step_roofline_frac": round(sb["step"] / (wall / args.steps) / 1e9 / PEAK_HBM_GBS, 4),
           "k_fcn2_frac": round(sb["pass2"] / p2_eval_s / 1e9 / PEAK_HBM_GBS, 4),
           "boundary_nodes": nbound, "exchange_bytes_per_dss": nbound * args.nz * 5 * 8,
           "finite": bool(torch.isfinite(V).all().item()), "launch_shape": shape}
    ctx.close()
    return out


def cpu_info():
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return model


def cpu_baseline(pkg, O, disc, phys, U0, Global, args, Ne):
    """The C oracle (the restated reference path; its results do not depend
    on the thread count) timed on the host: args.cpu_steps RW steps of the
    benchmark workload on every thread OpenMP is given (OMP_NUM_THREADS, else
    every core) and on one thread, and the reference's CPU configuration
    (ne=6, p=4, nz=10, 10 steps of 300 s) on both."""
    nall = O.set_threads(0)

    def timed(d, K, U, dt, steps, nt):
        O.set_threads(nt)
        orc = O.Oracle(d, phys, (K, K, K) if np.isscalar(K) else K)
        V = U.copy()
        t0 = time.perf_counter()
        orc.rw_step(V, dt, steps)
        return time.perf_counter() - t0

    hd = (Global.Model.HyperDCurl, Global.Model.HyperDGrad, Global.Model.HyperDDiv)
    tn = timed(disc, hd, U0, args.dt, args.cpu_steps, nall)
    # one thread: a bounded sample (one step at ne=60 is about 20 s)
    steps1 = max(1, args.cpu_steps // 3) if args.ne > 30 else args.cpu_steps
    t1 = timed(disc, hd, U0, args.dt, steps1, 1)
    d6 = pkg.discretization.build(6, args.p, 10, 30000.0)
    U6 = pkg.state.jet_state(d6, seed=0)
    K6 = pkg.host.hyperdiffusion_for(6)
    c1 = timed(d6, K6, U6, 300.0, 10, 1)
    cn = timed(d6, K6, U6, 300.0, 10, nall)
    O.set_threads(nall)
    ne6 = d6.nf * d6.N * d6.N * d6.nz
    rate = lambda pts, steps, t: round(pts * steps / t / 1e6, 4)  # noqa: E731
    return {"value": rate(Ne, args.cpu_steps, tn), "unit": "Mpts/s", "cores": nall, "kind": "port",
            "sample": f"{args.cpu_steps} RW step(s) of the C oracle (OpenMP, {nall} threads) on the same "
                      f"workload ({tn:.1f}s; {cpu_info()}, {os.cpu_count()} logical CPUs visible)",
            "single_core": {"value": rate(Ne, steps1, t1), "cores": 1, "steps": steps1, "seconds": round(t1, 2)},
            "cpu_config": {"workload": f"rw_step_fp64_ne6_p{args.p}_nz10, 10 steps, dt=300 s",
                           "mpts_s_1_core": rate(ne6, 10, c1), f"mpts_s_{nall}_threads": rate(ne6, 10, cn),
                           "seconds_1_core": round(c1, 3), f"seconds_{nall}_threads": round(cn, 3)}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--ne", type=int, default=60)
    ap.add_argument("--p", type=int, default=4)
    ap.add_argument("--nz", type=int, default=64)
    ap.add_argument("--dt", type=float, default=None,
                    help="default 100 s at ne<=30 and 3000/ne s above (horizontal acoustic CFL of p=4)")
    ap.add_argument("--hyperd", type=float, default=None, help="hyperviscosity coefficient (m^4/s)")
    ap.add_argument("--cpu-steps", type=int, default=3,
                    help="oracle RW steps for the CPU baseline on all threads, about 2 s each at ne=60 on 16 "
                         "threads; the one-thread sample runs a third of them (at least one) above ne=30 (0: skip)")
    ap.add_argument("--no-secondary", action="store_true",
                    help="skip the secondary FP64 drop-in line at ne=30 (dt=100 s)")
    ap.add_argument("--no-mixed", action="store_true", help="skip the mixed-precision comparison run")
    ap.add_argument("--no-share", action="store_true", help="skip the one-GPU-share run")
    ap.add_argument("--share-parts", type=int, default=8,
                    help="parts of the horizontal decomposition whose first part the share run steps")
    ap.add_argument("--no-ensemble", action="store_true", help="skip the batched-ensemble run")
    ap.add_argument("--no-autotune", action="store_true", help="keep the default launch shapes")
    ap.add_argument("--ntr", type=int, default=0, help="tracers in the FP64 state (reported in config)")
    ap.add_argument("--horlimit", action="store_true",
                    help="limited horizontal tracer transport (HorLimit; needs --ntr)")
    ap.add_argument("--no-adjoint", action="store_true", help="skip the adjoint gradient and its FD check")
    ap.add_argument("--adj-dirs", type=int, default=64, help="FD directions of the adjoint check")
    ap.add_argument("--only-adjoint", action="store_true",
                    help="run only the adjoint workload and print its JSON (not the benchmark line)")
    ap.add_argument("--only-ensemble", action="store_true",
                    help="run only the batched-ensemble workload and print its JSON (not the benchmark line)")
    ap.add_argument("--ens-members", type=int, default=32)
    ap.add_argument("--ens-steps", type=int, default=10)
    ap.add_argument("--ens-dt", type=float, default=150.0)
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MIB",
                    help="only run a plain device copy of MIB MiB three times (HBM counter calibration)")
    args = ap.parse_args()
    if args.dt is None:
        args.dt = 100.0 if args.ne <= 30 else 3000.0 / args.ne
    if args.horlimit and not args.ntr:
        ap.error("--horlimit needs tracers (--ntr)")
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}); "
              "the multi-GPU halo exchange is not implemented", file=sys.stderr)
        sys.exit(2)

    import torch

    import __graft_entry__ as ge

    if args.calibrate_copy:
        n = args.calibrate_copy * (1 << 20) // 8
        src = torch.ones(n, dtype=torch.float64, device="cuda:0")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"calibrate_copy_bytes": n * 8, "copies": 3}))
        return

    pkg = ge.load_package()
    if args.only_adjoint:  # profiling aid: the adjoint workload alone, its own JSON line
        print(json.dumps({"adjoint": adjoint(pkg, args)}), flush=True)
        return
    if args.only_ensemble:  # profiling aid: the ensemble workload alone, its own JSON line
        print(json.dumps({"ensemble": ensemble(pkg, args)}), flush=True)
        return
    host = pkg.host
    D = pkg.discretization
    t0 = time.perf_counter()
    disc = D.build(args.ne, args.p, args.nz, 30000.0)
    host_build_s = time.perf_counter() - t0
    phys = D.Phys()
    U0 = pkg.state.jet_state(disc, seed=0)
    if args.ntr:
        # tracers: mixing ratios 0.01 (1 + 0.1 k) of the density
        # (with --horlimit times 1.5 where |longitude| < 0.8, a step for the limiter to act on)
        shape_q = np.ones((1,) + U0.shape[1:])
        if args.horlimit:
            shape_q[0] += 0.5 * (np.abs(D.node_lonlat(disc)[:, 0]) < 0.8)[:, None]
        U0 = np.concatenate([U0] + [0.01 * (1 + 0.1 * k) * shape_q * U0[0:1] for k in range(args.ntr)], axis=0)
    print(f"[bench] setup ne={args.ne} p={args.p} nz={args.nz}: {host_build_s:.1f}s", file=sys.stderr, flush=True)
    # the same static inputs built by the device set-up kernels (numbering on the host)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    dev_build = host.device_build(args.ne, args.p, args.nz, 30000.0, device="cuda:0")
    torch.cuda.synchronize()
    device_build_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    g_native = host.cubed_sphere_native(args.ne, disc.rad)
    topo_s = time.perf_counter() - t0
    host.NumberingFemCGQuadGPU(g_native, args.p, device="cuda:0")
    torch.cuda.synchronize()
    numbering_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    pkg.grid.numbering_cg_quad(pkg.grid.cubed_sphere(args.ne, disc.rad), args.p)
    py_numbering_s = time.perf_counter() - t0
    setup = {"host_build_s": round(host_build_s, 3), "device_build_s": round(device_build_s, 3),
             "grid_and_numbering_s_of_device_build": round(numbering_s, 4),
             "grid_topology_s": round(topo_s, 4),
             "python_grid_and_numbering_s": round(py_numbering_s, 3),
             "what": "grid, numbering, metric (JacobiSphere3), DSS mass, layer sizes; device build = C++ "
                     "cubed-sphere topology on the host + numbering and set-up kernels on the device; the "
                     "host build and the Python grid/numbering are the restatement the tests check against"}
    del dev_build
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, hyperd=args.hyperd, device="cuda:0",
                                                          NumTr=args.ntr, horlimit=args.horlimit)
    ctx = host.init_context(FE, Metric, phys, Global)
    V = torch.as_tensor(U0, device="cuda:0").clone()
    shape = ctx.launch_shape()
    if not args.no_autotune:
        shape, _ = ctx.autotune(V, args.dt, Cache, JCache, reps=3)  # V is restored

    host.TimeStepper(V, args.dt, args.warmup, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    # timed region: one TimeStepper run of the steps (cgd_rw_run), HIP events
    # only around the fused tendency pass (each event is a stream barrier,
    # so the other passes are not bracketed here)
    ctx.profile(PASS2)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    host.TimeStepper(V, args.dt, args.steps, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    p2_ms, p2_launch = ctx.profile_read(1)
    finite = bool(torch.isfinite(V).all().item())
    V_fp64 = V.clone()  # warmup + steps from the initial state, for the mixed-precision comparison
    # per-pass breakdown from a few extra steps with every pass bracketed
    nb = min(args.steps, 5)
    ctx.profile(ALL_PASSES)
    host.TimeStepper(V, args.dt, nb, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    passes = {name: ctx.profile_read(i) for i, name in enumerate(("pass1", "pass2", "column"))}
    ctx.profile(0)
    print(f"[bench] {args.steps} steps in {wall:.3f}s, finite={finite}, pass2={p2_ms:.3f} ms, "
          f"breakdown over {nb} steps={passes}", file=sys.stderr, flush=True)

    sb = survey_bytes(args.ne, args.p, args.nz)
    Ne = sb["Ne"]
    ms_per_step = wall / args.steps * 1e3
    mpts = Ne * args.steps / wall / 1e6
    # dominant kernel: fused tendency pass (k_fcn2r; k_fcn2 where the metric
    # is not the same at all levels), 3 evaluations per step
    kern = "k_fcn2r" if ctx.info()[2] else "k_fcn2"
    n_eval = 3 * args.steps
    p2_eval_s = p2_ms / 1e3 / n_eval
    achieved = sb["pass2"] / p2_eval_s / 1e9
    workload = f"rw_step_fp64_ne{args.ne}_p{args.p}_nz{args.nz}" + (f"_tr{args.ntr}" if args.ntr else "") + (
        "_lim" if args.horlimit else "")
    traffic = measured_traffic(kern, workload, sb["pass2"])
    roofline = {"bound": "hbm", "kernel": f"{kern} (fused tendency pass)", "achieved": round(achieved, 1),
                "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(achieved / PEAK_HBM_GBS, 4),
                "traffic": traffic,
                "algorithmic_bytes_per_eval": sb["pass2"], "launches_per_eval": p2_launch // max(n_eval, 1),
                "ms_per_eval": round(p2_eval_s * 1e3, 4),
                "step_roofline_frac": round(sb["step"] / (wall / args.steps) / 1e9 / PEAK_HBM_GBS, 4),
                "pass_ms_per_step": {k: round(v[0] / nb, 4) for k, v in passes.items()}}
    # the committed kernel-trace summary of this workload: the same fraction
    # from rocprofv3's average dispatch duration of the kernel at this height
    tr = trace_average(f"{kern}<{args.p + 1}, {shape['chunk_levels']}", workload)
    if tr is not None:
        per_eval = roofline["launches_per_eval"] or 1
        roofline["trace"] = dict(tr, file=f"profiles/kernels_{workload}.json",
                                 frac_from_trace=round(sb["pass2"] / (tr["avg_us"] * per_eval * 1e3)
                                                       / PEAK_HBM_GBS, 4))

    mixed = None
    if not args.no_mixed and not args.ntr:
        mixed = mixed_precision(host, disc, phys, U0, args, ms_per_step, V_fp64)
        print(f"[bench] mixed precision: {mixed}", file=sys.stderr, flush=True)

    sec = None
    if not args.no_secondary and args.ne != 30 and not args.ntr:
        sec = secondary(pkg, args)
        print(f"[bench] secondary: {sec}", file=sys.stderr, flush=True)

    shr = None
    if not args.no_share and not args.ntr:
        shr = rank_share(pkg, args, disc)
        print(f"[bench] one GPU's share: {shr}", file=sys.stderr, flush=True)

    ens = None
    if not args.no_ensemble:
        ens = ensemble(pkg, args)
        print(f"[bench] ensemble: {ens}", file=sys.stderr, flush=True)

    adj = None
    if not args.no_adjoint:
        adj = adjoint(pkg, args)
        print(f"[bench] adjoint: {adj}", file=sys.stderr, flush=True)

    cpu = None
    if args.cpu_steps > 0 and not args.ntr:
        cpu = cpu_baseline(pkg, ge.load_oracle(), disc, phys, U0, Global, args, Ne)
        print(f"[bench] cpu baseline: {cpu}", file=sys.stderr, flush=True)

    out = {"metric": "RW step Mpts/s + % HBM roofline, FP64 vs FP32-mixed at stated err",
           "value": round(mpts, 2), "unit": "Mpts/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
           "ms_per_step": round(ms_per_step, 4), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
           "dtype": "f64", "data": "synthetic: seeded baroclinic jet (seed 0) on a flat cubed sphere",
           "config": {"workload": workload, "ne": args.ne, "p": args.p,
                      "nz": args.nz, "dt": args.dt, "hyperd": Global.Model.HyperDDiv, "points": Ne,
                      "precision": "fp64", "finite": finite, "tracers": args.ntr,
                      "horlimit": args.horlimit, "launch_shape": dict(shape, autotuned=not args.no_autotune)},
           "roofline": roofline, "cpu_baseline": cpu, "mixed": mixed, "ensemble": ens, "adjoint": adj,
           "secondary": sec, "one_gpu_share": shr, "setup": setup}
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
