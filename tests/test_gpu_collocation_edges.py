"""The collocation kernel bit for bit against the oracle at the ends of its
range (tests/collocation_edges.py)."""
import ctypes as C

import numpy as np
import pytest

from collocation_edges import KINDS, both_axes, faces
from gpu_helpers import qgrid, to_dev, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("ng,nx,ny", [(4, 13, 90), (3, 9, 90), (2, 9, 60)])
def test_collocation_bitwise(oracle, ng, nx, ny, kind):
    from quasar_amd import _lib
    torch, lib = torch_cuda(), _lib.load()
    rng = np.random.default_rng(ng * 10 + nx)
    along_x, along_y = both_axes(faces(kind, nx, ny, ng, rng), nx, ny, ng)
    for axis, (mx, my), f, cell in ((0, (nx, ny), along_x, oracle.cell_bx), (1, (ny, nx), along_y, oracle.cell_by)):
        og = oracle.grid(mx, my, ng)
        dev, out = to_dev([f, np.zeros(len(f))])
        torch.cuda.synchronize()
        _lib.check(lib.qmhd_collocate_face_to_cell(C.byref(qgrid(mx, my, ng)), axis, 0, C.c_void_p(dev.data_ptr()),
                                                   C.c_void_p(out.data_ptr()), None))
        torch.cuda.synchronize()
        want = np.array([cell(og, f, i, j, 0) for j in range(-ng, my + ng) for i in range(-ng, mx + ng)])
        np.testing.assert_array_equal(out.cpu().numpy(), want)
