"""The collocation of the step kernels, built for the host, bit for bit against
the oracle at the ends of its range (tests/collocation_edges.py)."""
import numpy as np
import pytest

from collocation_edges import KINDS, both_axes, faces
from host_kernels_ctypes import HostKernels


@pytest.fixture(scope="module")
def hk():
    import subprocess
    from host_kernels_ctypes import HOST_SO
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    return HostKernels()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("ng,nx,ny", [(4, 13, 90), (3, 9, 90), (2, 9, 60)])
def test_collocation_bitwise(oracle, hk, ng, nx, ny, kind):
    rng = np.random.default_rng(ng * 10 + nx)
    along_x, along_y = both_axes(faces(kind, nx, ny, ng, rng), nx, ny, ng)
    for axis, (mx, my), f, cell in ((0, (nx, ny), along_x, oracle.cell_bx), (1, (ny, nx), along_y, oracle.cell_by)):
        g = oracle.grid(mx, my, ng)
        got = hk.collocate(g, axis, 0, f)
        want = np.array([cell(g, f, i, j, 0) for j in range(-ng, my + ng) for i in range(-ng, mx + ng)])
        np.testing.assert_array_equal(got, want)
