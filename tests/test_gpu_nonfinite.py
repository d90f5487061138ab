"""Interface states beside damaged cells against the oracle: with a NaN or an
infinity in a cell of the interior the faces around it take the same path (MUSCL
or piecewise constant away from the cell, no finite states at it)."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import call, flags, ptrs, qgrid, scratch, to_dev, to_host, zeros_dev
from test_gpu_faces import G53, planes_of
from test_gpu_parity import face_mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("comp", [0, 2, 4, 7])
@pytest.mark.parametrize("order,ng", [(2, 2), (5, 3), (7, 4)])
def test_faces_beside_a_damaged_cell(oracle, order, ng, comp, bad):
    from quasar_amd import _lib
    lib = _lib.load()
    nx, ny = 37, 21
    g, qg = oracle.grid(nx, ny, ng), qgrid(nx, ny, ng)
    planes = planes_of("smooth", nx, ny, ng)
    oracle.fill_ghosts(g, (0, 0, 0, 0), (0, 0, 0, 0), planes)
    planes[comp].reshape(ny + 2 * ng, nx + 2 * ng)[ng + 9, ng + 17] = bad
    n = len(planes[0])
    sc = scratch(qg)
    for d in (0, 1):
        ref = [np.zeros(n) for _ in range(16)]
        oracle.reconstruct(g, d, order, (0, 0, 0, 0), G53, planes, ref)
        dev, out = to_dev(planes), zeros_dev(n, 16)
        call(lib.qmhd_reconstruct, C.byref(qg), d, order, flags((0, 0, 0, 0)), G53, ptrs(dev), ptrs(out),
             C.c_void_p(sc.data_ptr()), None)
        m = face_mask(nx, ny, ng, d)
        for c, (a, b) in enumerate(zip(to_host(out), ref)):
            a, b = a[m], b[m]
            np.testing.assert_array_equal(np.isfinite(a), np.isfinite(b), err_msg=f"dir {d} plane {c}")
            f = np.isfinite(b)
            assert np.all(np.abs(a[f] - b[f]) <= 1e-13 * np.maximum(1.0, np.abs(b[f]))), (d, c)
