#!/usr/bin/env python3
"""Zone-update throughput of the FP64 constrained-transport MHD step on one MI355X.

Workload: Orszag-Tang vortex, 2048^2 periodic cells on [0,1]^2, gamma 5/3,
rho = 25/(36 pi), p = 5/(12 pi), B0 = 1/sqrt(4 pi); MP7 characteristic
reconstruction + HLLD + upwind constrained transport, SSP-RK3, CFL 0.4 (0.2
effective for order >= 5), timestep from the device CFL reduction each step.
The state is seeded on the device from the closed-form initial condition and
stays resident in HBM; setup is outside the timed region.

One zone-update = one cell advanced by one full three-stage step, including
the CFL reduction, the positivity/solenoidality checks and the ghost fills
(python/quasar/mhd/cli.py:386-491 is the loop being timed).

Prints one JSON line.  `roofline` describes the kernel with the largest share
of the timed region: its average launch duration comes from HIP events that
the solver records around each launch on its own stream during the timed
steps.  `cpu_baseline` times the CPU restatement of the same step (OpenMP
C++) on a bounded sample of the same problem.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import pathlib
import sys
import time

ROOT = pathlib.Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

PEAK_HBM_GBS = 8000.0
PEAK_FP64_TFLOPS = 78.6

# Algorithmic cost per unit of each launch kind, FP64 MP7.  Units per launch
# are given by `units()`: one reconstruct launch covers the (n+1)(n+2ng) faces
# of each direction (the transverse quadrature needs the ghost rows), one flux
# launch the (n+1)^2 faces of each, corner the (n+1)^2 corners, cell_emf and
# update the n^2 cells, prep the (n+2ng)^2 padded cells.
#   bytes: every plane the kernel must read once and write once (8 B words),
#   flops: the arithmetic the algorithm needs for one unit (add, mul, div and
#          sqrt count 1, fma 2): the reference's operation sequence for that
#          unit, counting shared sub-results (a cell's x-direction point
#          recovery, used by seven stencil rows) once.
UNIT_COST = {
    # eigensystem 1.3k (0.7k of it the L R = I test), 8 projections 0.8k,
    # 14 MP7 face values + limiters 0.56k, back-projection 0.2k, checks 0.1k;
    # 8 state + 2 collocated field planes in, 16 interface planes + flag out
    "reconstruct": {"bytes": 8 * (8 + 2 + 16) + 4, "flops": 3000},
    # 16x4 point recoveries 0.9k, 4 HLLD solves 1.2k, admissibility and
    # wave speeds 0.4k; 16 interface planes in, 8 flux planes + rate out
    "flux": {"bytes": 8 * (16 + 8 + 1), "flops": 2500},
    # x-recovery 8x4x7 fma, y-recovery 4x4x8x7 fma, 16 EOS + E_z, Gauss
    # averages; 6 state + 2 collocated field planes in, cell E_z out
    "cell_emf": {"bytes": 8 * (6 + 2 + 1), "flops": 2600},
    # 11 eight-tap edge interpolations; 2 flux, cell E_z, 2 flag planes in, E_z out
    "corner": {"bytes": 8 * (3 + 1) + 2 * 4, "flops": 180},
    # flux difference, curl, Shu-Osher combine; 8 base + 8 stage + 2x8 flux +
    # E_z planes in, 8 planes out
    "update": {"bytes": 8 * (8 + 8 + 16 + 1 + 8), "flops": 90},
    # two correctly rounded 8-tap collocations, theta and checks; 8 candidate
    # planes in (the base only where a check is close), 2 collocated planes out
    "prep": {"bytes": 8 * (8 + 2), "flops": 1000},
}
NG = 4


def parse():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--n", type=int, default=2048, help="cells per side")
    ap.add_argument("--cpu-seconds", type=float, default=15.0,
                    help="bound on the CPU baseline's timed work")
    ap.add_argument("--cpu-n", type=int, default=1024, help="cells per side of the CPU sample")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-forms", action="store_true", help="skip the FP32 and FP32+learned runs")
    ap.add_argument("--no-target", action="store_true",
                    help="skip the target block (Orszag-Tang 4096^2 + 1e-3 noise, 500 steps, every form)")
    ap.add_argument("--target-n", type=int, default=4096)
    ap.add_argument("--target-steps", type=int, default=500)
    ap.add_argument("--profile-steps", type=int, default=6,
                    help="steps of the separate pass with per-launch HIP events that times the kernels")
    ap.add_argument("--autotune", type=int, default=0, metavar="STEPS",
                    help="autotune every solver's launch shapes over STEPS steps per candidate before timing")
    ap.add_argument("--only-form", choices=("fp32", "fp32_learned"),
                    help="time only this form (the line's value and kernel shares are that form's; for profiling)")
    ap.add_argument("--sweep", action="store_true",
                    help="instead of the single-run benchmark: the batched sweep of 64 mixed-size runs "
                         "(FP32 + learned, one graph launch per step, autotuned launch shapes)")
    ap.add_argument("--sweep-runs", type=int, default=64)
    ap.add_argument("--sweep-sizes", default="256,384,512,768,1024",
                    help="comma-separated run sizes the sweep draws from")
    ap.add_argument("--sweep-seq-steps", type=int, default=30,
                    help="steps per run of the run-by-run comparison of the sweep")
    ap.add_argument("--problem", choices=("orszag_tang", "rotor"), default="orszag_tang",
                    help="workload: the Orszag-Tang vortex (periodic) or the MHD rotor (gamma 1.4, disk rho 10 "
                         "spinning at omega 20 with a taper to r 0.115, Bx 5/sqrt(4 pi), outflow)")
    ap.add_argument("--noise", type=float, default=0.0,
                    help="seeded white-noise amplitude on rho (relative), vx and vy (the 4096^2 deck uses 1e-3)")
    ap.add_argument("--copy-probe-mib", type=int, default=0,
                    help="before the timed region, copy a buffer of this size once (HBM traffic calibration "
                         "for counter runs)")
    ap.add_argument("--summarize-flops", metavar="PMC_DIR",
                    help="no run: turn a rocprofv3 --pmc output of the FP64 F64 VALU instruction counters "
                         "(SQ_INSTS_VALU_ADD_F64, _MUL_F64, _FMA_F64, _TRANS_F64) into FP64 operations per launch "
                         "per kernel kind, written to profiles/flops_ot<n>_mp7.json")
    ap.add_argument("--summarize-counters", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="no run: turn two rocprofv3 --pmc outputs (FETCH_SIZE, WRITE_SIZE) of a run made with "
                         "--copy-probe-mib into HBM bytes per launch per kernel kind, written to "
                         "profiles/traffic_ot<n>_mp7.json")
    return ap.parse_args()


def orszag_tang(n: int, noise: float = 0.0):
    from quasar_amd import mhd
    spec = mhd.MhdInitialConditionSpec()
    spec.kind = "orszag_tang"
    spec.grid = mhd.Grid2D(n, n, 1.0, 1.0, 0.0, 0.0, 4)
    spec.gamma = 5.0 / 3.0
    spec.b_uniform = [1.0 / math.sqrt(4.0 * math.pi), 0.0, 0.0]
    spec.ot_rho = 25.0 / (36.0 * math.pi)
    spec.ot_p = 5.0 / (12.0 * math.pi)
    spec.noise_amplitude = noise
    spec.noise_seed = 0
    return spec


AUTOTUNE_STEPS = 0
PROBLEM = "orszag_tang"


def make_solver(n: int, arithmetic: str = "fp64", indicator: str = "none", noise: float = 0.0,
                problem: str = "orszag_tang"):
    from quasar_amd import batch, mhd
    if problem == "rotor":
        spec, sides = batch.problem("rotor", n, noise, 0)
    else:
        spec, sides = orszag_tang(n, noise), "periodic"
    cfg = mhd.MhdConfig()
    cfg.grid = spec.grid
    cfg.gamma = spec.gamma
    cfg.reconstruction = "mp7"
    cfg.arithmetic = arithmetic
    cfg.indicator = indicator
    cfg.cfl = 0.4
    cfg.boundary.set_fluid_all(sides)
    cfg.boundary.set_field_all(sides)
    solver = mhd.MhdSolver2D(cfg)
    state = mhd.build_initial_state(spec)
    for name, plane in state.items():
        solver.seed_state(name, plane)
    if indicator == "mlp":
        from quasar_amd import learned
        params, threshold, _ = learned.load()
        solver.set_indicator(params, threshold)
    if AUTOTUNE_STEPS > 0:
        tuning = solver.autotune(AUTOTUNE_STEPS)
        print(f"bench: autotuned {arithmetic}/{indicator}: {tuning}", file=sys.stderr, flush=True)
    return solver


STATE_NAMES = ("rho", "mx", "my", "mz", "energy", "bx_face", "by_face", "bz_cell")
GROUPS = ((0,), (1, 2, 3), (1, 2, 3), (1, 2, 3), (4,), (5, 6, 7), (5, 6, 7), (5, 6, 7))


def interior_state(solver, n: int):
    import numpy as np
    return [np.asarray(solver.state_component_to_host(nm)).reshape(n + 2 * NG, n + 2 * NG)[NG:NG + n, NG:NG + n]
            for nm in STATE_NAMES]


def rel_l1_by_variable(got, ref):
    """Per-variable relative L1 against the variable's own L1 norm; a minor
    momentum or field component (own norm below 1e-2 of its vector's, e.g. mz
    and bz in 2-D problems) against its vector's norm."""
    import numpy as np
    out = {}
    for c, nm in enumerate(STATE_NAMES):
        own = float(np.abs(ref[c]).sum())
        group = max(float(np.abs(ref[k]).sum()) for k in GROUPS[c])
        denom = own if own >= 1e-2 * group else group
        out[nm] = float(np.abs(got[c] - ref[c]).sum()) / denom
    return out


def timed_run(solver, steps: int):
    import torch
    solver.synchronize()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    done, sim_t = solver.run(steps)
    solver.synchronize()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    if done != steps:
        raise RuntimeError(f"run stopped after {done} of {steps} steps")
    return wall, sim_t


def sweep(args) -> dict:
    """Batched sweep: FP32 + learned runs advanced together by one graph launch
    per step, in both batched forms (each run's step on its own stream; the
    tile work queue over all runs' tiles), against the same runs stepped one
    after another, and against the FP64 plain form (batched) for throughput
    and, at each learned run's end time, for the per-run error."""
    import numpy as np
    from quasar_amd import batch
    sizes = tuple(int(v) for v in args.sweep_sizes.split(","))
    descs = batch.sweep_runs(args.sweep_runs, seed=0, sizes=sizes)
    cells = sum(d["n"] ** 2 for d in descs)
    print(f"bench: sweep of {len(descs)} runs, {cells} cells, building FP32+learned runs (autotuned)",
          file=sys.stderr, flush=True)
    runs, tuned = batch.build_sweep(descs, "fp32", "mlp", autotune_steps=2)
    b = batch.Batch(runs)
    b.run(args.warmup)
    before = [b.status(k) for k in range(len(descs))]
    t0 = time.perf_counter()
    b.run(args.steps)
    wall = time.perf_counter() - t0
    status = [b.status(k) for k in range(len(descs))]
    rejected = sum(st["rejected"] - st0["rejected"] for st, st0 in zip(status, before))
    fatal = sum(1 for st in status if st["fatal"])
    accepted = sum(d["n"] ** 2 * (st["accepted"] - st0["accepted"]) for d, st, st0 in zip(descs, status, before))
    stream_value = accepted / wall
    del b
    print(f"bench: batched (one stream per run) {args.steps} steps in {wall:.3f} s", file=sys.stderr, flush=True)
    # The same runs through the tile work queue: one launch shape for every
    # run (the largest size's), the workgroups per queue launch autotuned.
    q_runs, q_tuned = batch.build_sweep(descs, "fp32", "mlp", autotune_steps=2, shared_tuning=True)
    qb = batch.Batch(q_runs, queue=True)
    queue_blocks = qb.autotune(2)
    qb.run(args.warmup)
    q_before = [qb.status(k) for k in range(len(descs))]
    t0 = time.perf_counter()
    qb.run(args.steps)
    q_wall = time.perf_counter() - t0
    q_status = [qb.status(k) for k in range(len(descs))]
    q_accepted = sum(d["n"] ** 2 * (st["accepted"] - st0["accepted"])
                     for d, st, st0 in zip(descs, q_status, q_before))
    rejected += sum(st["rejected"] - st0["rejected"] for st, st0 in zip(q_status, q_before))
    fatal += sum(1 for st in q_status if st["fatal"])
    queue_value = q_accepted / q_wall
    del qb, q_runs
    print(f"bench: batched (tile work queue, {queue_blocks} workgroups per launch) {args.steps} steps in "
          f"{q_wall:.3f} s", file=sys.stderr, flush=True)
    value = max(stream_value, queue_value)
    # Run-by-run comparison (each run's own loop, one after another).
    seq_runs, _ = batch.build_sweep(descs, "fp32", "mlp")
    for s_, d in zip(seq_runs, descs):
        s_.set_tuning(tuned[d["n"]])
        s_.run(1)
    t0 = time.perf_counter()
    for s_ in seq_runs:
        s_.run(args.sweep_seq_steps)
    for s_ in seq_runs:
        s_.synchronize()
    seq_wall = time.perf_counter() - t0
    seq_value = cells * args.sweep_seq_steps / seq_wall
    del seq_runs
    print(f"bench: run-by-run {args.sweep_seq_steps} steps in {seq_wall:.3f} s", file=sys.stderr, flush=True)
    # FP64 plain form of every run, batched, one step fewer than the learned
    # runs took; each then steps on its own to its learned run's end time.
    ref_runs, _ = batch.build_sweep(descs, "fp64", "none")
    rb = batch.Batch(ref_runs)
    rb.run(args.warmup)
    t0 = time.perf_counter()
    rb.run(args.steps - 1)
    ref_wall = time.perf_counter() - t0
    ref_elapsed = [rb.status(k)["sim_time"] for k in range(len(descs))]
    del rb
    fp64_stream_value = cells * (args.steps - 1) / ref_wall
    # The FP64 form through the tile work queue as well (timing only): the
    # comparison takes each form's faster batch.
    fq_runs, _ = batch.build_sweep(descs, "fp64", "none", autotune_steps=2, shared_tuning=True)
    fqb = batch.Batch(fq_runs, queue=True)
    fqb.autotune(2)
    fqb.run(args.warmup)
    t0 = time.perf_counter()
    fqb.run(args.steps - 1)
    fq_wall = time.perf_counter() - t0
    del fqb, fq_runs
    fp64_queue_value = cells * (args.steps - 1) / fq_wall
    fp64_value = max(fp64_stream_value, fp64_queue_value)
    print(f"bench: FP64 batched {args.steps - 1} steps: {ref_wall:.3f} s (streams), {fq_wall:.3f} s (queue)",
          file=sys.stderr, flush=True)
    l1 = []
    for s_, r_, d, st, t64 in zip(runs, ref_runs, descs, status, ref_elapsed):
        n = d["n"]
        remaining = st["sim_time"] - t64
        if not remaining > 0:
            # The FP64 run took larger steps and is past the learned run's
            # end time: a fresh FP64 run goes there on its own.
            (r_,), _ = batch.build_sweep([d], "fp64", "none")
            remaining = st["sim_time"]
        done, t_ = r_.run(100 * (args.steps + args.warmup), remaining)
        if t_ != remaining:
            raise RuntimeError(f"sweep run {d['run']}: the FP64 run stopped after {done} steps, t = {t_}")
        got, exp = _interior(s_, n), _interior(r_, n)
        l1.append(rel_l1_by_variable(got, exp))
    rho = np.array([e["rho"] for e in l1])
    worst = np.array([max(e.values()) for e in l1])
    kinds = [d["kind"] for d in descs]
    by_kind = {}
    for kind in sorted(set(kinds)):
        sel = np.array([k == kind for k in kinds])
        by_kind[kind] = {"rho_median": float(np.median(rho[sel])), "rho_max": float(rho[sel].max()),
                         "any_variable_max": float(worst[sel].max())}
    return {
        "metric": "zone-updates/s, batched sweep of independent runs on 1 MI355X (FP32 + learned)",
        "value": round(value, 1), "unit": "zone-updates/s", "n_gpus": 1, "runs": len(descs), "cells": cells,
        "steps": args.steps, "warmup": args.warmup,
        "wall_s": round(q_wall if queue_value >= stream_value else wall, 4),
        "accepted_zone_updates": q_accepted if queue_value >= stream_value else accepted,
        "rejected_steps": rejected, "fatal_runs": fatal,
        "batched_form": "tile work queue" if queue_value >= stream_value else "one stream per run",
        "stream_batch_value": round(stream_value, 1), "queue_batch_value": round(queue_value, 1),
        "queue_blocks": queue_blocks, "queue_tuning": next(iter(q_tuned.values())),
        "run_by_run_value": round(seq_value, 1), "batching_gain": round(value / seq_value, 3),
        "fp64_batched_value": round(fp64_value, 1),
        "fp64_stream_batch_value": round(fp64_stream_value, 1), "fp64_queue_batch_value": round(fp64_queue_value, 1),
        "speedup_vs_fp64_batched": round(value / fp64_value, 3),
        "rel_l1_vs_fp64_at_equal_time": {"rho_median": float(np.median(rho)), "rho_max": float(rho.max()),
                                         "any_variable_max": float(worst.max()), "by_kind": by_kind},
        "sizes": {str(n): sum(1 for d in descs if d["n"] == n) for n in sorted({d["n"] for d in descs})},
        "tuning": {str(k): v for k, v in tuned.items()},
        "data": "synthetic: seeded Orszag-Tang and rotor initial conditions with 1e-3 white noise",
    }


def _interior(solver, n: int):
    import numpy as np
    return [np.asarray(solver.state_component_to_host(nm)).reshape(n + 2 * NG, n + 2 * NG)[NG:NG + n, NG:NG + n]
            for nm in STATE_NAMES]


def units(kind: str, n: int) -> int:
    if kind == "reconstruct":
        return 2 * (n + 1) * (n + 2 * NG)
    if kind == "flux":
        return 2 * (n + 1) * (n + 1)
    if kind == "corner":
        return (n + 1) * (n + 1)
    if kind == "prep":
        return (n + 2 * NG) * (n + 2 * NG)
    return n * n


def roofline(times: dict, n: int):
    """The dominant kernel kind's roofline from its launch times (HIP events
    on the solver stream, a profiled pass after the timed region).  Its FP64
    operations per launch are the counted ones (rocprofv3 F64 VALU
    instruction counters, profiles/flops_ot<n>_mp7.json) when that summary
    exists for this size, else the per-unit estimate of UNIT_COST."""
    kind = max((k for k in UNIT_COST), key=lambda k: times[k][0])
    total_ms, launches = times[kind]
    avg_s = total_ms / launches / 1e3
    cost = UNIT_COST[kind]
    u = units(kind, n)
    bytes_alg = cost["bytes"] * u
    counted = counted_flops(kind, n)
    flops = counted if counted is not None else cost["flops"] * u
    gbs = bytes_alg / avg_s / 1e9
    tfs = flops / avg_s / 1e12
    balance = PEAK_FP64_TFLOPS * 1e12 / (PEAK_HBM_GBS * 1e9)
    if flops / bytes_alg > balance:
        r = {"bound": "fp64_valu", "achieved": round(tfs, 3), "peak": PEAK_FP64_TFLOPS, "unit": "TFLOP/s",
             "frac": round(tfs / PEAK_FP64_TFLOPS, 4)}
    else:
        r = {"bound": "hbm", "achieved": round(gbs, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
             "frac": round(gbs / PEAK_HBM_GBS, 4)}
    r["traffic"] = measured_traffic(kind, n)
    r["kernel"] = kind
    r["avg_launch_ms"] = round(total_ms / launches, 4)
    r["launches"] = launches
    r["algorithmic_bytes_per_launch"] = bytes_alg
    r["flops_per_launch"] = flops
    r["flops_basis"] = ("counted: 64 lanes x (ADD + MUL + TRANS + 2 FMA) F64 VALU instructions per launch, "
                        "rocprofv3 on this kernel" if counted is not None else "per-unit estimate (UNIT_COST)")
    r["flops_estimate_per_launch"] = cost["flops"] * u
    r["hbm_frac_algorithmic"] = round(gbs / PEAK_HBM_GBS, 4)
    r["bound_note"] = ("the kernel runs on the FP64 vector pipe (VALU); MI355X's FP64 vector and matrix peak are "
                       "both 78.6 TFLOP/s")
    shares = {k: round(v[0], 3) for k, v in times.items()}
    return r, shares


def counted_flops(kind: str, n: int):
    """FP64 operations per launch of a kernel kind from the committed counter
    summary (Orszag-Tang runs only)."""
    p = ROOT / "profiles" / f"flops_ot{n}_mp7.json"
    if PROBLEM != "orszag_tang" or not p.exists():
        return None
    try:
        return json.loads(p.read_text()).get(kind)
    except (ValueError, OSError):
        return None


def measured_traffic(kind: str, n: int):
    """HBM bytes per launch from the committed counter summary, when one exists
    for this kernel and size (Orszag-Tang runs only)."""
    p = ROOT / "profiles" / f"traffic_ot{n}_mp7.json"
    if PROBLEM != "orszag_tang" or not p.exists():
        return None
    try:
        data = json.loads(p.read_text())
        return data.get(kind)
    except (ValueError, OSError):
        return None


# Kernels of each timed kind of the FP64 MP7 step (one dispatch of each per
# launch of the kind).  A symbol matches every instantiation whose name
# contains it; their per-dispatch values are averaged.
KERNEL_SYMBOLS = {
    "prep": ("prep_kernel<true, 8>",),
    "reconstruct": ("reconstruct_kernel_queue<double, 7>", "reconstruct_fallback_kernel_queue<double, 7>"),
    "flux": ("flux_kernel_queue<double, 7, false>",),
    "cell_emf": ("cell_emf_kernel<double, 7, false, 16, 16>",),
    "corner": ("corner_tiled_kernel<double, 7>",),
    "update": ("update_kernel<double>",),
}


def _counter_rows(run_dir: str, counter: str):
    """(kernel name, value) of every dispatch's `counter` in a rocprofv3 --pmc
    csv output directory."""
    import csv
    import glob
    rows = []
    for path in glob.glob(os.path.join(run_dir, "**", "*counter_collection.csv"), recursive=True):
        with open(path, newline="") as f:
            for row in csv.DictReader(f):
                if row.get("Counter_Name") == counter:
                    rows.append((row["Kernel_Name"], float(row["Counter_Value"])))
    return rows


def _means(rows):
    sums, counts = {}, {}
    for name, v in rows:
        sums[name] = sums.get(name, 0.0) + v
        counts[name] = counts.get(name, 0) + 1
    return {k: sums[k] / counts[k] for k in sums}


F64_COUNTERS = ("SQ_INSTS_VALU_ADD_F64", "SQ_INSTS_VALU_MUL_F64", "SQ_INSTS_VALU_FMA_F64", "SQ_INSTS_VALU_TRANS_F64")


def summarize_flops(pmc_dir: str) -> dict:
    """FP64 operations per launch of each kernel kind: the F64 VALU
    instruction counts (per wave, summed over the dispatch) times the 64 lanes
    of a wave, an FMA counting two operations."""
    means = {c: _means(_counter_rows(pmc_dir, c)) for c in F64_COUNTERS}
    names = set().union(*(m.keys() for m in means.values()))
    out = {"unit": "FP64 operations per launch",
           "rule": "64 x (ADD_F64 + MUL_F64 + TRANS_F64 + 2 FMA_F64), counters summed over a dispatch"}
    per_kernel = {}
    for nm in names:
        add, mul, fma, trans = (means[c].get(nm, 0.0) for c in F64_COUNTERS)
        per_kernel[nm] = 64.0 * (add + mul + trans + 2.0 * fma)
    out["kernels"] = {k: round(v) for k, v in sorted(per_kernel.items())}
    for kind, syms in KERNEL_SYMBOLS.items():
        vals = [_matching_mean(per_kernel, sym) for sym in syms]
        if any(v is None for v in vals):
            continue
        out[kind] = round(sum(vals))
    return out


def _matching_mean(per_kernel: dict, sym: str):
    vals = [v for k, v in per_kernel.items() if sym in k]
    return sum(vals) / len(vals) if vals else None


def summarize_counters(fetch_dir: str, write_dir: str, n: int, probe_mib: int) -> dict:
    """HBM bytes per launch of each kernel kind.  FETCH_SIZE and WRITE_SIZE read
    KiB per dispatch; each is scaled by the factor that makes the copy probe
    (the largest copy dispatch: probe_mib MiB read and written once) count
    exactly its size."""
    frows = _counter_rows(fetch_dir, "FETCH_SIZE")
    wrows = _counter_rows(write_dir, "WRITE_SIZE")
    fprobe = max((v for k, v in frows if "copy" in k.lower()), default=0.0)
    wprobe = max((v for k, v in wrows if "copy" in k.lower()), default=0.0)
    if fprobe <= 0 or wprobe <= 0:
        raise RuntimeError("no copy-probe dispatch in the counter output")
    probe_kib = probe_mib * 1024.0
    fetch_scale, write_scale = probe_kib / fprobe, probe_kib / wprobe
    fetch, write = _means(frows), _means(wrows)
    out = {"probe_mib": probe_mib, "probe_fetch_kib": fprobe, "probe_write_kib": wprobe,
           "fetch_scale": fetch_scale, "write_scale": write_scale, "unit": "bytes per launch"}
    for kind, syms in KERNEL_SYMBOLS.items():
        fvals = [_matching_mean(fetch, sym) for sym in syms]
        wvals = [_matching_mean(write, sym) for sym in syms]
        if any(v is None for v in fvals):
            continue
        fb = sum(fvals) * fetch_scale * 1024.0
        wb = sum(v or 0.0 for v in wvals) * write_scale * 1024.0
        out[kind] = round(fb + wb)
        out[kind + "_fetch_bytes"] = round(fb)
        out[kind + "_write_bytes"] = round(wb)
    return out


def cpu_model() -> str:
    try:
        for line in pathlib.Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(n: int, budget_s: float):
    """The CPU restatement (OpenMP C++) on Orszag-Tang n^2 MP7 FP64, the
    benchmark's workload on a smaller grid: whole steps are taken until
    `budget_s` seconds of CPU work have been timed (at least one)."""
    sys.path.insert(0, str(ROOT / "tests"))
    from oracle_ctypes import Oracle, OracleSolver, ic_spec
    oracle = Oracle()
    g = oracle.grid(n, n, 4)
    spec = ic_spec("orszag_tang", 5.0 / 3.0, b_uniform=[1 / math.sqrt(4 * math.pi), 0, 0],
                   ot_rho=25 / (36 * math.pi), ot_p=5 / (12 * math.pi))
    status, planes = oracle.seed(g, spec)
    if status != 0:
        raise RuntimeError("oracle seed failed")
    ref = OracleSolver(oracle, g, 5.0 / 3.0, 0.4, 7)
    ref.seed(planes)
    steps = 0
    t0 = time.perf_counter()
    while True:
        ref.step(ref.cfl_limit())
        steps += 1
        el = time.perf_counter() - t0
        if el >= budget_s or steps >= 1000:
            break
    cores = int(os.environ.get("OMP_NUM_THREADS", "0")) or len(os.sched_getaffinity(0))
    return {"value": round(n * n * steps / el, 1), "unit": "zone-updates/s", "cores": cores, "kind": "port",
            "cpu_model": cpu_model(),
            "sample": f"Orszag-Tang {n}^2 MP7+HLLD+CT FP64, {steps} step(s) ({el:.1f} s), C++ restatement "
                      f"with OpenMP on {cores} host threads"}


def main():
    global AUTOTUNE_STEPS, PROBLEM
    args = parse()
    AUTOTUNE_STEPS = args.autotune
    PROBLEM = args.problem
    if args.summarize_flops:
        summary = summarize_flops(args.summarize_flops)
        path = ROOT / "profiles" / f"flops_ot{args.n}_mp7.json"
        path.write_text(json.dumps(summary, indent=1) + "\n")
        print(json.dumps(summary))
        return
    if args.summarize_counters:
        summary = summarize_counters(args.summarize_counters[0], args.summarize_counters[1], args.n,
                                     args.copy_probe_mib or 1024)
        path = ROOT / "profiles" / f"traffic_ot{args.n}_mp7.json"
        path.write_text(json.dumps(summary, indent=1) + "\n")
        print(json.dumps(summary))
        return
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}, WORLD_SIZE {world}); "
              "the step is not sharded across GPUs", file=sys.stderr)
        sys.exit(2)

    import torch
    if not torch.cuda.is_available():
        print("bench.py: no HIP device visible", file=sys.stderr)
        sys.exit(1)
    torch.cuda.set_device(0)
    from quasar_amd import _lib
    _lib.load()  # raises when the gfx950 library is missing: there is no CPU path

    if args.sweep:
        print(json.dumps(sweep(args)), flush=True)
        return
    n = args.n
    if args.only_form:
        arith, ind = ("fp32", "none") if args.only_form == "fp32" else ("fp32", "mlp")
        print(f"bench: seeding {PROBLEM} {n}^2 MP7, form {args.only_form}", file=sys.stderr, flush=True)
        s = make_solver(n, arith, ind, args.noise, PROBLEM)
        if args.warmup > 0:
            s.run(args.warmup)
        s.set_profiling(True)
        w, st = timed_run(s, args.steps)
        times = s.kernel_times()
        print(json.dumps({"form": args.only_form, "value": round(n * n * args.steps / w, 1), "unit": "zone-updates/s",
                          "ms_per_step": round(w / args.steps * 1e3, 4), "steps": args.steps, "warmup": args.warmup,
                          "sim_time": st, "kernel_ms": {k: round(v[0], 3) for k, v in times.items()}}), flush=True)
        return
    print(f"bench: seeding {PROBLEM} {n}^2 MP7 FP64", file=sys.stderr, flush=True)
    solver = make_solver(n, noise=args.noise, problem=PROBLEM)
    if args.copy_probe_mib > 0:
        a = torch.ones(args.copy_probe_mib * (1 << 20) // 8, dtype=torch.float64, device="cuda")
        b = torch.empty_like(a)
        b.copy_(a)
        torch.cuda.synchronize()
        del a, b
    t_warm = 0.0
    if args.warmup > 0:
        t_warm = solver.run(args.warmup)[1]
    print(f"bench: warmup {args.warmup} steps done", file=sys.stderr, flush=True)

    # Every form is timed with per-launch profiling off; the kernel times of
    # the roofline come from a separate profiled pass afterwards.
    wall, sim_t = timed_run(solver, args.steps)
    done = args.steps
    t_ref = t_warm + sim_t
    ref_state = interior_state(solver, n) if not args.no_forms else None
    solver.set_profiling(True)
    solver.run(args.profile_steps)
    roof, shares = roofline(solver.kernel_times(), n)
    solver.set_profiling(False)
    del solver
    print(f"bench: {done} steps, wall {wall:.3f} s; profiled pass of {args.profile_steps} steps: kernels "
          f"{sum(shares.values()) / 1e3:.3f} s", file=sys.stderr, flush=True)

    zone_updates = n * n * done
    value = zone_updates / wall
    line = {
        "metric": "zone-updates/s, 1 MI355X: FP64 plain vs FP32+learned at fixed L1 err; %HBM",
        "value": round(value, 1),
        "unit": "zone-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall / done * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": f"synthetic: {'Orszag-Tang' if PROBLEM == 'orszag_tang' else 'rotor'} initial condition from "
                "its closed form" +
                (f" plus seeded white noise of amplitude {args.noise:g} on rho, vx, vy" if args.noise else ""),
        "config": {"workload": f"{PROBLEM}_{n}x{n}_mp7_hlld_ct_ssprk3_fp64", "form": "plain FP64",
                   "cfl": 0.4, "boundaries": "periodic" if PROBLEM == "orszag_tang" else "outflow",
                   "sim_time": t_ref, "noise": args.noise},
        "hbm_frac_step": round(value * 512 / (PEAK_HBM_GBS * 1e9), 5),
        "kernel_ms_profiled_pass": shares,
        "roofline": roof,
    }
    if not args.no_forms:
        line["forms"] = forms_to_time(n, args.noise, args.warmup, t_ref, ref_state, wall / done)
        del ref_state
    if not args.no_target:
        line["target"] = target_block(args)
    if not args.no_cpu_baseline:
        print("bench: timing the CPU baseline", file=sys.stderr, flush=True)
        line["cpu_baseline"] = cpu_baseline(args.cpu_n, args.cpu_seconds)
    else:
        line["cpu_baseline"] = None
    print(json.dumps(line), flush=True)


FORMS = (("fp32", "fp32", "none"), ("fp32_learned", "fp32", "mlp"))


def forms_to_time(n: int, noise: float, warmup: int, t_ref: float, ref_state, fp64_s_per_step: float,
                  forms=FORMS) -> dict:
    """Each form from the same seed, warmed up like the FP64 run, then timed
    (profiling off) through its auto-dt loop to the FP64 run's end time (its
    last step clipped onto it), and compared with the FP64 state there."""
    out = {}
    for name, arith, ind in forms:
        print(f"bench: {name} form {n}^2 to t = {t_ref:.6g}", file=sys.stderr, flush=True)
        s = make_solver(n, arith, ind, noise, PROBLEM)
        t_w = s.run(warmup)[1] if warmup > 0 else 0.0
        if ind == "mlp":
            s.plain_faces()
        w, steps, t_end = timed_run_to(s, t_ref - t_w)
        per_step = w / steps
        entry = {
            "value": round(n * n * steps / w, 1),
            "ms_per_step": round(per_step * 1e3, 4),
            "steps": steps,
            "speedup_vs_fp64": round(fp64_s_per_step / per_step, 3),
            "sim_time": t_w + t_end,
            "rel_l1_vs_fp64": rel_l1_by_variable(interior_state(s, n), ref_state),
        }
        if ind == "mlp":
            plain, total = s.plain_faces()
            entry["plain_face_share"] = round(plain / max(total, 1), 5)
        out[name] = entry
        del s
    return out


def timed_run_to(solver, t_end: float, max_steps: int = 1_000_000):
    """The auto-dt loop until the simulated time reaches t_end."""
    import torch
    solver.synchronize()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    done, sim_t = solver.run(max_steps, t_end)
    solver.synchronize()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    if sim_t != t_end:
        raise RuntimeError(f"run stopped at t = {sim_t} before {t_end}")
    return wall, done, sim_t


def target_block(args) -> dict:
    """The accuracy-throughput target: Orszag-Tang target_n^2 with seeded 1e-3
    white noise on rho, vx, vy.  FP64 plain runs target_steps steps; the FP32
    and FP32+learned forms run from the same seed to the same simulated time;
    all three are timed with profiling off.  Each form's per-variable
    relative L1 distance from the FP64 state is reported; the target is
    >= 3x the FP64 zone-updates/s at density L1 <= 1e-4."""
    global PROBLEM
    saved, PROBLEM = PROBLEM, "orszag_tang"
    try:
        n, steps, noise, warm = args.target_n, args.target_steps, 1e-3, 2
        print(f"bench: target block, FP64 {n}^2, {steps} steps", file=sys.stderr, flush=True)
        s = make_solver(n, noise=noise)
        t_w = s.run(warm)[1]
        w, t = timed_run(s, steps)
        ref = interior_state(s, n)
        del s
        t_ref = t_w + t
        forms = forms_to_time(n, noise, warm, t_ref, ref, w / steps)
        del ref
        learned = forms["fp32_learned"]
        return {
            "workload": f"orszag_tang_{n}x{n}_noise1e-3_mp7_hlld_ct_ssprk3",
            "fp64": {"value": round(n * n * steps / w, 1), "ms_per_step": round(w / steps * 1e3, 4),
                     "steps": steps, "warmup": warm, "sim_time": t_ref},
            "forms": forms,
            "learned_speedup_vs_fp64": learned["speedup_vs_fp64"],
            "learned_rho_rel_l1": learned["rel_l1_vs_fp64"]["rho"],
            "target_met": bool(learned["speedup_vs_fp64"] >= 3.0 and learned["rel_l1_vs_fp64"]["rho"] <= 1e-4),
            "note": "forms compared at the FP64 run's simulated time; every run timed with profiling off",
        }
    finally:
        PROBLEM = saved


if __name__ == "__main__":
    main()
