"""A batched run that stops says why, in a warning of the call and afterwards:
the check that its own loop would have failed, and after how many steps.  The
other runs of the batch take their steps."""
import warnings

import pytest

pytestmark = pytest.mark.gpu


def runs():
    from quasar_amd import batch
    ds = [{"run": k, "n": n, "kind": "orszag_tang", "noise": 1e-3, "noise_seed": k} for k, n in enumerate((48, 32, 40))]
    return batch.build_sweep(ds, "fp64", "none")[0]


def spoil(solver, fault):
    w = 40
    if fault == "divergence":
        bx = solver.state_component_to_host("bx_face").reshape(w, w).copy()
        bx[4 + 7, 4 + 9] += 0.1
        solver.seed_state("bx_face", bx)
    else:
        en = solver.state_component_to_host("energy").reshape(w, w).copy()
        en[4 + 7, 4 + 9] = 1e-3
        solver.seed_state("energy", en)


@pytest.mark.parametrize("fault,words", [("divergence", "divergence-free"), ("pressure", "not admissible")])
@pytest.mark.parametrize("queue", [False, True])
def test_a_stopped_run_says_why(queue, fault, words):
    from quasar_amd import batch
    solvers = runs()
    spoil(solvers[1], fault)
    b = batch.Batch(solvers, queue=queue)
    with pytest.warns(RuntimeWarning, match=f"batch run 1 stopped after 0 accepted steps.*{words}"):
        b.run(3)
    assert words in b.failure(1) and b.failure(0) == b.failure(2) == ""
    assert [b.status(k)["accepted"] for k in range(3)] == [3, 0, 3]
    assert [b.status(k)["fatal"] for k in range(3)] == [False, True, False]
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        b.run(2)  # told once
    assert b.status(0)["accepted"] == 5


def test_a_run_whose_controller_fails_says_so():
    """A rejected step is finished by the run's own positivity controller; what
    that raises is the run's failure."""
    from quasar_amd import batch
    from test_gpu_batch import low_pressure_muscl_run
    solvers = [low_pressure_muscl_run()]
    b = batch.Batch(solvers)
    solvers[0].fail_after_pieces(0)
    with pytest.warns(RuntimeWarning, match="injected integrator failure"):
        b.run(12)
    assert b.status(0)["fatal"] and "injected" in b.failure(0)


def test_a_batch_without_failures_stays_silent():
    from quasar_amd import batch
    b = batch.Batch(runs())
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        b.run(3)
    assert [b.failure(k) for k in range(3)] == ["", "", ""]
