"""The autotuner times only the knobs that shape a launch of the run's scheme:
MP5/MP7 take their fluxes in fixed tiles, so their flux block stays as set."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [(64, 1), (16, 16)])
@pytest.mark.parametrize("arithmetic,indicator", [("fp64", "none"), ("fp32", "mlp")])
def test_autotune_leaves_a_knob_without_effect(arithmetic, indicator, block):
    from quasar_amd import batch
    d = [{"run": 0, "n": 64, "kind": "orszag_tang", "noise": 1e-3, "noise_seed": 5}]
    (s,), _ = batch.build_sweep(d, arithmetic, indicator)
    s.set_tuning({**s.tuning(), "flux_block_x": block[0], "flux_block_y": block[1]})
    choice = s.autotune(1)
    assert (choice["flux_block_x"], choice["flux_block_y"]) == block
    assert s.run(2)[0] == 2
