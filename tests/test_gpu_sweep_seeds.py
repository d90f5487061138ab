"""Queued sweeps of 24 small learned runs (64^2 to 128^2, Orszag-Tang and rotor
alternating) over a dozen noise seeds: every run takes the steps it was asked
for, none is rejected or stopped, and each ends bit for bit where its own loop
ends.

The launches of a batch share the device between runs, and a run's step
status, its checks and its face-list counters are written by blocks on all
eight XCDs.  A run whose checks or counters went wrong stops early or takes
other faces through the general path; either shows here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ("rho", "mx", "my", "mz", "energy", "bx_face", "by_face", "bz_cell")
STEPS = (8, 5)  # both register parities end a call


@pytest.mark.parametrize("seed", range(12))
def test_queued_sweep_ends_where_the_own_loops_end(seed):
    from quasar_amd import batch, learned
    p, t, _ = learned.load()
    descs = [{"run": k, "n": (64, 96, 128)[(k + seed) % 3], "kind": ("orszag_tang", "rotor")[k % 2], "noise": 1e-3,
              "noise_seed": 1000 * (seed + 1) + k} for k in range(24)]
    queued, _ = batch.build_sweep(descs, "fp32", "mlp", (p, t))
    alone, _ = batch.build_sweep(descs, "fp32", "mlp", (p, t))
    print(f"queued sweep, seed {seed}", flush=True)
    b = batch.Batch(queued, queue=True)
    for n in STEPS:
        b.run(n)
    for k, s in enumerate(alone):
        done, time = s.run(sum(STEPS))
        assert done == sum(STEPS)
        assert b.status(k) == {"accepted": done, "rejected": 0, "fatal": False, "sim_time": time}, (descs[k], b.status(k))
        for name in NAMES:
            np.testing.assert_array_equal(queued[k].state_component_to_host(name), s.state_component_to_host(name),
                                          err_msg=f"{descs[k]} {name}")
