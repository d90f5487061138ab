"""The indicator's gradient over the sizes and chunkings where its waves share a
partial differently (chunks 1: a partial per wave; 2 and 3: two waves; more:
four), down to a single sample, against the oracle's at the bound of the other
gradient tests."""
import numpy as np
import pytest

from test_gpu_learned import BLOCKS, gpu_grad, random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("n", [1, 16, 65, 1003])
def test_gradient_for_every_sharing(oracle, n, chunks):
    params, x, y, w = random_problem(13 + n, n)
    loss, grad = gpu_grad(params, x, y, w, chunks)
    exp_loss, exp = oracle.mlp_loss_grad(params, x, y, w, bf16=True)
    assert abs(loss - exp_loss) <= 2e-3 * abs(exp_loss)
    for name, (a, b) in BLOCKS.items():
        norm = np.linalg.norm(exp[a:b])
        assert np.linalg.norm(grad[a:b] - exp[a:b]) <= 2e-3 * max(norm, 1e-6), (name, n, chunks)
