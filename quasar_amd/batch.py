"""Batched runs: many independent MHD runs advanced by one HIP graph launch per
step (include/quasar_mhd.h, qmhd_batch_*), and the seeded sweep of mixed-size
Orszag-Tang and rotor runs used as the batched workload.

Each run keeps its own solver (buffers sized for its grid).  The batch
captures the auto-dt step of every run, each on the run's own stream forked
from one master stream, into a graph; the accept/reject decision of each
run's step is made on the device, so the graph replays without host
synchronization.  Runs of the same size share one autotuned launch shape
(qmhd_solver_autotune on the first run of that size).
"""
from __future__ import annotations

import ctypes as C
import math
import warnings
from typing import Dict, List, Sequence

import numpy as np

from . import _lib, mhd

SWEEP_SIZES = (256, 384, 512, 768, 1024)


class Batch:
    """Graph-captured stepping of independent solvers (they stay owned by the
    caller and must be stepped only through the batch while it exists).

    queue=False: each run's step on its own stream inside one graph.
    queue=True: the tile work queue, one launch per step phase over the tiles
    of every run (the runs must share scheme, form and launch shapes);
    queue_blocks is the number of workgroups per queue launch (0: one per
    tile), which autotune() can pick."""

    def __init__(self, solvers: Sequence["mhd.MhdSolver2D"], queue: bool = False, queue_blocks: int = 0):
        self._lib = _lib.load()
        self._solvers = list(solvers)
        self.queue = bool(queue)
        self._told = set()
        arr = (C.c_void_p * len(self._solvers))(*[s._h.value for s in self._solvers])
        h = C.c_void_p()
        if self.queue:
            _lib.check(self._lib.qmhd_batch_create_queued(arr, len(self._solvers), int(queue_blocks), C.byref(h)))
        else:
            _lib.check(self._lib.qmhd_batch_create(arr, len(self._solvers), C.byref(h)))
        self._h = h

    def autotune(self, trial_steps: int = 3) -> int:
        """Queue mode: the fastest workgroups-per-launch candidate over
        trial_steps steps (every run is put back in its state)."""
        best = C.c_int()
        _lib.check(self._lib.qmhd_batch_autotune(self._h, int(trial_steps), C.byref(best)))
        return best.value

    def __del__(self):
        h = getattr(self, "_h", None)
        if h:
            self._lib.qmhd_batch_destroy(h)
            self._h = None

    def run(self, steps: int) -> None:
        """Advance every run by `steps`; a run that stops on the way is told
        in a RuntimeWarning (the other runs take their steps)."""
        before = self._lib.qmhd_batch_fatal_runs(self._h)
        _lib.check(self._lib.qmhd_batch_run(self._h, int(steps)))
        if self._lib.qmhd_batch_fatal_runs(self._h) != before:
            for k in range(len(self._solvers)):
                why = self.failure(k)
                if why and k not in self._told:
                    self._told.add(k)
                    warnings.warn(f"batch run {k} stopped {why}", RuntimeWarning, stacklevel=2)

    def failure(self, run: int) -> str:
        """Why run `run` stopped, or "" where it has not."""
        return self._lib.qmhd_batch_run_failure(self._h, int(run)).decode()

    def status(self, run: int) -> Dict:
        a, r = C.c_int64(), C.c_int64()
        fatal, t = C.c_int(), C.c_double()
        _lib.check(self._lib.qmhd_batch_run_status(self._h, int(run), C.byref(a), C.byref(r), C.byref(fatal),
                                                   C.byref(t)))
        return {"accepted": a.value, "rejected": r.value, "fatal": bool(fatal.value), "sim_time": t.value}


def sweep_runs(count: int = 64, seed: int = 0, sizes=SWEEP_SIZES) -> List[Dict]:
    """The seeded sweep: sizes drawn uniformly from `sizes` with a Philox
    generator keyed by `seed`, Orszag-Tang and rotor alternating, each with a
    seeded 1e-3 white-noise perturbation of rho, vx and vy (noise seed = run
    index)."""
    r = np.random.Generator(np.random.Philox(key=seed))
    picks = r.integers(0, len(sizes), size=count)
    return [{"run": k, "n": int(sizes[int(picks[k])]), "kind": "orszag_tang" if k % 2 == 0 else "rotor",
             "noise": 1e-3, "noise_seed": k} for k in range(count)]


def problem(kind: str, n: int, noise: float, noise_seed: int):
    """(MhdInitialConditionSpec, boundary) of one sweep run."""
    spec = mhd.MhdInitialConditionSpec()
    spec.kind = kind
    spec.grid = mhd.Grid2D(n, n, 1.0, 1.0, 0.0, 0.0, 4)
    if kind == "orszag_tang":
        spec.gamma = 5.0 / 3.0
        spec.b_uniform = [1.0 / math.sqrt(4.0 * math.pi), 0.0, 0.0]
        spec.ot_rho = 25.0 / (36.0 * math.pi)
        spec.ot_p = 5.0 / (12.0 * math.pi)
        sides = "periodic"
    else:
        spec.gamma = 1.4
        spec.center = [0.5, 0.5]
        spec.b_uniform = [5.0 / math.sqrt(4.0 * math.pi), 0.0, 0.0]
        spec.p_ambient = 1.0
        sides = "outflow"
    spec.noise_amplitude = noise
    spec.noise_seed = noise_seed
    return spec, sides


def make_run(desc: Dict, arithmetic: str = "fp32", indicator: str = "mlp", network=None):
    spec, sides = problem(desc["kind"], desc["n"], desc["noise"], desc["noise_seed"])
    cfg = mhd.MhdConfig()
    cfg.grid = spec.grid
    cfg.gamma = spec.gamma
    cfg.reconstruction = "mp7"
    cfg.arithmetic = arithmetic
    cfg.indicator = indicator
    cfg.boundary.set_fluid_all(sides)
    cfg.boundary.set_field_all(sides)
    s = mhd.MhdSolver2D(cfg)
    for name, plane in mhd.build_initial_state(spec).items():
        s.seed_state(name, plane)
    if indicator == "mlp":
        params, threshold = network
        s.set_indicator(params, threshold)
    return s


def build_sweep(descs: Sequence[Dict], arithmetic: str = "fp32", indicator: str = "mlp", network=None,
                autotune_steps: int = 0, shared_tuning: bool = False):
    """Solvers of the sweep; with autotune_steps > 0, the first run of each
    size is autotuned and the others of that size take its launch shape.
    shared_tuning: the first run of the largest size is autotuned and every
    run takes its launch shape (the tile work queue needs one shape for all
    runs); the returned dict then maps every size to that one tuning."""
    if indicator == "mlp" and network is None:
        from . import learned
        p, t, _ = learned.load()
        network = (p, t)
    solvers, tuned = [], {}
    if shared_tuning and autotune_steps > 0 and descs:
        largest = max(range(len(descs)), key=lambda k: descs[k]["n"])
        solvers = [make_run(d, arithmetic, indicator, network) for d in descs]
        common = solvers[largest].autotune(autotune_steps)
        for s in solvers:
            s.set_tuning(common)
        return solvers, {d["n"]: common for d in descs}
    for d in descs:
        s = make_run(d, arithmetic, indicator, network)
        if autotune_steps > 0:
            if d["n"] not in tuned:
                tuned[d["n"]] = s.autotune(autotune_steps)
            else:
                s.set_tuning(tuned[d["n"]])
        solvers.append(s)
    return solvers, tuned
