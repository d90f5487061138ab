"""Cell E_z where waves march far: the kernel walks two or four times as many
rows per wave once that leaves 512 blocks, so the grids of the oracle tests
never take those paths.  Here they are held bit for bit to the short march (the
one that the oracle tests check) on windows of the same data, thin states
included, whose points' pressures are decided again after the march; and to each
other over the tile shapes, whose waves march 8 to 32 rows."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import call, flags, ptrs, qgrid, scratch, to_dev, zeros_dev
from test_gpu_faces import G53, planes_of

pytestmark = pytest.mark.gpu

PERIODIC = (0, 0, 0, 0)


def blocks(nx, ny, march):
    return -(-(nx + 1) // 16) * -(-(ny + 1) // (16 * march))


def cell_ez(lib, nx, ny, ng, order, dev):
    import torch
    from quasar_amd import _lib
    qg = qgrid(nx, ny, ng)
    n = (nx + 2 * ng) * (ny + 2 * ng)
    faces = zeros_dev(n, 32)
    out, eq = zeros_dev(n, 3), zeros_dev(n, 2)
    tables = _lib.QEmfTables(*[t.data_ptr() for t in out], *[t.data_ptr() for t in eq])
    sc = scratch(qg)
    call(lib.qmhd_ct_emf_prepare, C.byref(qg), order, 0, flags(PERIODIC), G53, ptrs(dev), ptrs(faces[:16]),
         ptrs(faces[16:]), C.byref(tables), C.c_void_p(sc.data_ptr()), None)
    torch.cuda.synchronize()
    return out[0].reshape(ny + 2 * ng, nx + 2 * ng)


@pytest.mark.parametrize("state", ["smooth", "thin"])
@pytest.mark.parametrize("order,ng", [(5, 3), (7, 4)])
@pytest.mark.parametrize("nx,ny,march", [(603, 451, 2), (1003, 701, 4)])
def test_far_marches_match_the_short_one(oracle, nx, ny, march, order, ng, state):
    from quasar_amd import _lib
    lib = _lib.load()
    assert [m for m in (4, 2, 1) if m == 1 or blocks(nx, ny, m) >= 512][0] == march
    planes = planes_of("smooth", nx, ny, ng)
    if state == "thin":
        kinetic = sum(planes[c] ** 2 for c in (1, 2, 3)) / (2 * planes[0])
        planes[4] = kinetic + 0.5 * sum(planes[c] ** 2 for c in (5, 6, 7)) + \
            0.3 * np.random.default_rng(3).random(len(kinetic))
    oracle.fill_ghosts(oracle.grid(nx, ny, ng), PERIODIC, PERIODIC, planes)
    dev = to_dev(planes)
    far = cell_ez(lib, nx, ny, ng, order, dev)
    # Columns over the whole height and rows over the whole width, about the
    # edges of waves, blocks and the grid.
    for i0, wx, j0, wy in ((0, 40, 0, ny), (nx - 37, 37, 0, ny), (481, 33, 0, ny), (0, nx, 0, 30), (0, nx, ny - 75, 75)):
        assert blocks(wx, wy, 2) < 512
        cut = (slice(j0, j0 + wy + 2 * ng), slice(i0, i0 + wx + 2 * ng))
        window = [p.reshape(ny + 2 * ng, nx + 2 * ng)[cut].contiguous().reshape(-1) for p in dev]
        near = cell_ez(lib, wx, wy, ng, order, window)
        # (At a cut the window's outer collocated cells take one-sided closures.)
        inner = (slice(ng if j0 == 0 else 2 * ng, ng + wy if j0 + wy == ny else wy),
                 slice(ng if i0 == 0 else 2 * ng, ng + wx if i0 + wx == nx else wx))
        np.testing.assert_array_equal(far[cut][inner].cpu().numpy(), near[inner].cpu().numpy(), err_msg=f"{i0} {j0}")


@pytest.mark.parametrize("scheme,ng", [("mp5", 3), ("mp7", 4)])
@pytest.mark.parametrize("arithmetic", ["fp64", "fp32"])
def test_tile_shapes_give_the_same_bits(scheme, ng, arithmetic):
    """16 x 16, 32 x 8 and 8 x 32 cells, four times as many rows each."""
    from quasar_amd import mhd
    nx, ny = 1003, 701
    planes = planes_of("smooth", nx, ny, ng)
    names = ("rho", "mx", "my", "mz", "energy", "bx_face", "by_face", "bz_cell")
    want = None
    for tile in (0, 1, 2):
        cfg = mhd.MhdConfig()
        cfg.grid = mhd.Grid2D(nx, ny, 1.0, 0.7, 0.0, 0.0, ng)
        cfg.gamma = G53
        cfg.reconstruction = scheme
        cfg.arithmetic = arithmetic
        cfg.boundary.set_fluid_all("outflow")
        cfg.boundary.set_field_all("outflow")
        s = mhd.MhdSolver2D(cfg)
        s.set_tuning({**s.tuning(), "emf_tile": tile})
        for name, plane in zip(names, planes):
            # A uniform field in the plane: any state may be seeded with it.
            s.seed_state(name, np.full_like(plane, 0.4) if name in ("bx_face", "by_face") else plane)
        assert s.run(1)[0] == 1
        got = [s.state_component_to_host(name) for name in names]
        want = want or got
        for name, a, b in zip(names, got, want):
            np.testing.assert_array_equal(a, b, err_msg=f"tile {tile} {name}")
