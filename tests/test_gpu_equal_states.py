"""Equal states give equal cell E_z to the last bit, whichever rule a cell takes:
the quadrature, or the cell average where a point of its stencil is not
admissible.  The corner's one-dimensional shortcuts compare across such
borders."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import call, flags, ptrs, qgrid, scratch, to_dev, to_host, zeros_dev
from test_gpu_faces import G53

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,ng", [(5, 3), (7, 4)])
def test_cell_ez_across_rules(order, ng):
    from quasar_amd import _lib
    lib = _lib.load()
    nx, ny = 37, 29
    qg = qgrid(nx, ny, ng)
    h = 2 if order == 5 else 3
    w, n = nx + 2 * ng, (nx + 2 * ng) * (ny + 2 * ng)
    rng = np.random.default_rng(order)
    sc = scratch(qg)
    for _ in range(12):
        rho, p = rng.uniform(0.3, 3, 2)
        v, b = rng.normal(size=3), rng.normal(size=3)
        en = p / (G53 - 1) + 0.5 * rho * v @ v + 0.5 * b @ b
        planes = [np.full(n, q) for q in (rho, *(rho * v), en, *b)]
        bad = (ng + 13) * w + ng + 17
        planes[4][bad] = -100 * en  # no point of the cells around it is admissible, or few
        dev, faces = to_dev(planes), zeros_dev(n, 32)
        out, eq = zeros_dev(n, 3), zeros_dev(n, 2)
        tables = _lib.QEmfTables(*[t.data_ptr() for t in out], *[t.data_ptr() for t in eq])
        f = (0, 0, 0, 0)
        for d in (0, 1):
            call(lib.qmhd_reconstruct, C.byref(qg), d, order, flags(f), G53, ptrs(dev), ptrs(faces[16 * d:16 * d + 16]),
                 C.c_void_p(sc.data_ptr()), None)
        call(lib.qmhd_ct_emf_prepare, C.byref(qg), order, 0, flags(f), G53, ptrs(dev), ptrs(faces[:16]), ptrs(faces[16:]),
             C.byref(tables), C.c_void_p(sc.data_ptr()), None)
        ez = to_host(out[:1])[0].reshape(ny + 2 * ng, w)[ng:ng + ny, ng:ng + nx]
        near = np.zeros((ny, nx), dtype=bool)
        near[13 - h:13 + h + 1, 17 - h:17 + h + 1] = True
        assert len(np.unique(ez[~near])) == 1
        near[13, 17] = False
        np.testing.assert_array_equal(ez[near], ez[0, 0])
