"""The collocation kernel bit for bit against the oracle where its sums and
quotients are decided: exact ties (integers, dyadic samples), near-ties, the
bottom of the exponent range, exact zeros and cancelling samples, at every
window width and on grids with no cell outside the ghost closures' reach."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import qgrid, to_dev, torch_cuda

pytestmark = pytest.mark.gpu


def faces(data, n, rng):
    if data == "integers":
        return rng.integers(-1000, 1000, n).astype(float)
    if data == "dyadic":
        return rng.integers(-8, 8, n) * 2.0 ** rng.integers(-30, 30, n)
    if data == "thirds":
        return np.where(rng.random(n) < 0.2, 2.0 / 3.0, 1.0 / 3.0)
    if data == "tiny":
        return rng.normal(size=n) * 1e-300
    if data == "zeros":
        return np.where(rng.random(n) < 0.9, 0.0, rng.normal(size=n))
    return rng.normal(size=n) * 10.0 ** rng.integers(-12, 12, size=n)


@pytest.mark.parametrize("data", ["integers", "dyadic", "thirds", "tiny", "zeros", "scales"])
@pytest.mark.parametrize("ng,nx,ny", [(4, 70, 9), (4, 1, 3), (3, 11, 67), (2, 33, 5), (1, 7, 6)])
def test_collocation_bitwise(oracle, ng, nx, ny, data):
    from quasar_amd import _lib
    torch, lib = torch_cuda(), _lib.load()
    rng = np.random.default_rng(100 * ng + nx)
    g, og = qgrid(nx, ny, ng), oracle.grid(nx, ny, ng)
    n = (nx + 2 * ng) * (ny + 2 * ng)
    face = faces(data, n, rng)
    dev, out = to_dev([face, np.zeros(n)])
    for axis, cell in ((0, oracle.cell_bx), (1, oracle.cell_by)):
        for co in (0, 1):
            torch.cuda.synchronize()
            _lib.check(lib.qmhd_collocate_face_to_cell(C.byref(g), axis, co, C.c_void_p(dev.data_ptr()),
                                                       C.c_void_p(out.data_ptr()), None))
            torch.cuda.synchronize()
            want = [cell(og, face, i, j, co) for j in range(-ng, ny + ng) for i in range(-ng, nx + ng)]
            np.testing.assert_array_equal(out.cpu().numpy(), np.array(want))
