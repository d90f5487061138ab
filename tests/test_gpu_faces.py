"""MP5/MP7 interface states, face fluxes and cell E_z against the oracle around
the edges of the kernels' tiles (64 x 4 and 32 x 8 faces, 16 x 16 and 32 x 8
fluxes, 16 columns by 4 to 16 rows of cell E_z, and the halos they stage), on smooth states, on states at rest with no
transverse field, on supersonic ones and on ones far from unit density.  The
bound is the one every launch of the ABI is held to: 1e-13 relative L1."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import call, flags, ptrs, qgrid, rel_l1_state, scratch, to_dev, to_host, zeros_dev
from test_gpu_parity import face_mask, flux_mask

pytestmark = pytest.mark.gpu
G53 = 5.0 / 3.0


def planes_of(state, nx, ny, ng):
    rng = np.random.default_rng(1000 * nx + ny)
    shape = (ny + 2 * ng, nx + 2 * ng)
    y, x = np.mgrid[0:shape[0], 0:shape[1]]
    w = lambda a, b: np.sin(2 * np.pi * (x / 17.0 + a)) * np.cos(2 * np.pi * (y / 13.0 + b))
    rho, p = 1 + 0.3 * w(0.1, 0.2), 1 + 0.4 * w(0.3, 0.7)
    v = [0.5 * w(0.2, 0.9), 0.4 * w(0.6, 0.1), 0.3 * w(0.8, 0.4)]
    b = [0.6 + 0.2 * w(0.5, 0.5), 0.3 * w(0.4, 0.6), 0.2 * w(0.9, 0.3)]
    if state == "at_rest":
        v = [0 * rho] * 3
        b = [0.75 + 0 * rho, 0 * rho, 0 * rho]
        rho = np.where(x > shape[1] // 2, 0.125, 1.0)
        p = np.where(x > shape[1] // 2, 0.1, 1.0)
    elif state == "supersonic":
        v = [8 * q for q in v]
        rho = rho * np.where(rng.random(shape) < 0.1, 4.0, 1.0)
    elif state == "dense":
        rho, p = 1e4 * rho, 1e2 * p
    en = p / (G53 - 1) + 0.5 * rho * sum(q * q for q in v) + 0.5 * sum(q * q for q in b)
    return [np.ascontiguousarray(q).ravel() for q in (rho, *(rho * q for q in v), en, *b)]


def compare(got, want, sides, what):
    """NaN (faces no fallback makes admissible) at the same entries; the rest to the bound."""
    finite = np.ones(len(want[0]), dtype=bool)
    for a, b in zip(got, want):
        np.testing.assert_array_equal(np.isfinite(a), np.isfinite(b))
        finite &= np.isfinite(b)
    got, want = [q[finite] for q in got], [q[finite] for q in want]
    for side in sides:
        for c in range(8):
            assert rel_l1_state(got, want, c, side) <= 1e-13, (*what, side + c)


@pytest.mark.parametrize("state", ["smooth", "at_rest", "supersonic", "dense"])
@pytest.mark.parametrize("order,ng,nx,ny", [(7, 4, 15, 17), (7, 4, 63, 4), (7, 4, 65, 31), (5, 3, 31, 9), (5, 3, 64, 3),
                                            (5, 4, 33, 32), (7, 4, 5, 8)])
def test_faces_at_tile_edges(oracle, order, ng, nx, ny, state):
    from quasar_amd import _lib
    lib = _lib.load()
    g, qg = oracle.grid(nx, ny, ng), qgrid(nx, ny, ng)
    planes = planes_of(state, nx, ny, ng)
    oracle.fill_ghosts(g, (0, 0, 0, 0), (0, 0, 0, 0), planes)
    n = len(planes[0])
    sc = scratch(qg)
    for d in (0, 1):
        ref16, ref8 = [np.zeros(n) for _ in range(16)], [np.zeros(n) for _ in range(8)]
        oracle.reconstruct(g, d, order, (0, 0, 0, 0), G53, planes, ref16)
        dev, out = to_dev(planes), zeros_dev(n, 16)
        call(lib.qmhd_reconstruct, C.byref(qg), d, order, flags((0, 0, 0, 0)), G53, ptrs(dev), ptrs(out),
             C.c_void_p(sc.data_ptr()), None)
        m = face_mask(nx, ny, ng, d)
        got, want = [q[m] for q in to_host(out)], [q[m] for q in ref16]
        compare(got, want, (0, 8), ("state", d))
        oracle.face_flux(g, d, order, 0, (0, 0, 0, 0), G53, ref16, ref8)
        dev, out = to_dev(ref16), zeros_dev(n, 8)
        call(lib.qmhd_hlld_flux, C.byref(qg), d, order, 0, flags((0, 0, 0, 0)), G53, ptrs(dev), ptrs(out),
             C.c_void_p(sc.data_ptr()), None)
        m = flux_mask(nx, ny, ng)
        got, want = [q[m] for q in to_host(out)], [q[m] for q in ref8]
        compare(got, want, (0,), ("flux", d))


@pytest.mark.parametrize("state", ["smooth", "at_rest", "supersonic", "dense", "thin"])
@pytest.mark.parametrize("ng,nx,ny,sides", [(2, 63, 5, (0, 0, 0, 0)), (2, 33, 17, (1, 1, 1, 1)), (4, 65, 8, (2, 2, 0, 0)),
                                            (3, 5, 31, (1, 2, 2, 1))])
def test_muscl_faces_at_tile_edges(oracle, ng, nx, ny, sides, state):
    """`thin` holds states whose pressure is near or below zero: the faces there
    take the fallback chain, which the oracle's NaN pattern and values show."""
    from quasar_amd import _lib
    lib = _lib.load()
    g, qg = oracle.grid(nx, ny, ng), qgrid(nx, ny, ng)
    planes = planes_of("smooth" if state == "thin" else state, nx, ny, ng)
    if state == "thin":
        kinetic = sum(planes[c] ** 2 for c in (1, 2, 3)) / (2 * planes[0])
        rng = np.random.default_rng(3)
        planes[4] = kinetic + 0.5 * sum(planes[c] ** 2 for c in (5, 6, 7)) + 0.1 * rng.random(len(kinetic))
    oracle.fill_ghosts(g, sides, sides, planes)
    n = len(planes[0])
    sc = scratch(qg)
    for d in (0, 1):
        ref16 = [np.zeros(n) for _ in range(16)]
        oracle.reconstruct(g, d, 2, sides, G53, planes, ref16)
        dev, out = to_dev(planes), zeros_dev(n, 16)
        call(lib.qmhd_reconstruct, C.byref(qg), d, 2, flags(sides), G53, ptrs(dev), ptrs(out), C.c_void_p(sc.data_ptr()),
             None)
        m = face_mask(nx, ny, ng, d)
        compare([q[m] for q in to_host(out)], [q[m] for q in ref16], (0, 8), ("muscl", d))


@pytest.mark.parametrize("state", ["smooth", "at_rest", "supersonic", "dense", "thin"])
@pytest.mark.parametrize("order,ng,nx,ny,sides", [(7, 4, 15, 17, 0), (7, 4, 16, 3, 1), (7, 4, 33, 64, 0), (5, 3, 31, 9, 1),
                                                  (5, 3, 17, 16, 0), (7, 4, 18, 5, 1), (7, 4, 5, 8, 0)])
def test_cell_ez_at_tile_edges(oracle, order, ng, nx, ny, sides, state):
    """`thin` holds points of zero and negative pressure: those cells take the
    cell-average E_z, and the decision is the oracle's."""
    from quasar_amd import _lib
    lib = _lib.load()
    g, qg = oracle.grid(nx, ny, ng), qgrid(nx, ny, ng)
    F = (sides,) * 4
    planes = planes_of("smooth" if state == "thin" else state, nx, ny, ng)
    if state == "thin":
        kinetic = sum(planes[c] ** 2 for c in (1, 2, 3)) / (2 * planes[0])
        rng = np.random.default_rng(3)
        planes[4] = kinetic + 0.5 * sum(planes[c] ** 2 for c in (5, 6, 7)) + 0.3 * rng.random(len(kinetic))
    oracle.fill_ghosts(g, F, F, planes)
    n = len(planes[0])
    ref16 = [[np.zeros(n) for _ in range(16)] for _ in range(2)]
    for d in (0, 1):
        oracle.reconstruct(g, d, order, F, G53, planes, ref16[d])
    want = oracle.ct_emf(g, order, 0, F, G53, planes, *ref16)["cell_ez"]
    dev, faces = to_dev(planes), zeros_dev(n, 32)
    out, eq = zeros_dev(n, 3), zeros_dev(n, 2)
    tables = _lib.QEmfTables(*[t.data_ptr() for t in out], *[t.data_ptr() for t in eq])
    sc = scratch(qg)
    for d in (0, 1):
        call(lib.qmhd_reconstruct, C.byref(qg), d, order, flags(F), G53, ptrs(dev), ptrs(faces[16 * d:16 * d + 16]),
             C.c_void_p(sc.data_ptr()), None)
    call(lib.qmhd_ct_emf_prepare, C.byref(qg), order, 0, flags(F), G53, ptrs(dev), ptrs(faces[:16]), ptrs(faces[16:]),
         C.byref(tables), C.c_void_p(sc.data_ptr()), None)
    m = np.zeros((ny + 2 * ng, nx + 2 * ng), dtype=bool)
    m[ng:ng + ny + (sides != 0), ng:ng + nx + (sides != 0)] = True
    got, ref = to_host(out[:1])[0][m.ravel()], want[m.ravel()]
    scale = np.abs(ref).sum()
    assert np.abs(got - ref).sum() <= 1e-13 * max(scale, 1e-3 * len(ref)), (np.abs(got - ref).max(), scale)


@pytest.mark.parametrize("data", ["smooth", "x_only", "y_only", "uniform"])
@pytest.mark.parametrize("order,ng,nx,ny,sides", [(7, 4, 15, 17, (0, 0, 0, 0)), (7, 4, 40, 33, (1, 1, 0, 0)),
                                                  (7, 4, 16, 9, (2, 2, 2, 2)), (5, 3, 47, 16, (1, 1, 1, 1)),
                                                  (5, 4, 31, 5, (0, 0, 2, 1)), (7, 4, 5, 48, (1, 2, 0, 0))])
def test_corner_at_tile_edges(oracle, order, ng, nx, ny, sides, data):
    """Corner E_z over 16 x 16 blocks that hold the boundary, with data whose
    one-dimensional shortcuts are taken everywhere, in places and nowhere; the
    bound is the one of the launches above."""
    from quasar_amd import _lib
    lib = _lib.load()
    g, qg = oracle.grid(nx, ny, ng), qgrid(nx, ny, ng)
    planes = [p.reshape(ny + 2 * ng, nx + 2 * ng).copy() for p in planes_of("smooth", nx, ny, ng)]
    if data in ("x_only", "uniform"):
        planes = [np.broadcast_to(p[:1], p.shape).copy() for p in planes]
    if data in ("y_only", "uniform"):
        planes = [np.broadcast_to(p[:, :1], p.shape).copy() for p in planes]
    if data == "x_only":
        planes[5][:] = planes[5][0, 0]
    if data == "y_only":
        planes[6][:] = planes[6][0, 0]
    planes = [p.ravel() for p in planes]
    oracle.fill_ghosts(g, sides, sides, planes)
    n = len(planes[0])
    i16, f8 = [[np.zeros(n) for _ in range(16)] for _ in range(2)], [[np.zeros(n) for _ in range(8)] for _ in range(2)]
    for d in (0, 1):
        oracle.reconstruct(g, d, order, sides, G53, planes, i16[d])
        oracle.face_flux(g, d, order, 0, sides, G53, i16[d], f8[d])
    want = oracle.ct_emf(g, order, 0, sides, G53, planes, *i16)["ez"]
    dev = [to_dev(x) for x in (planes, *i16, *f8)]
    ez, sc = zeros_dev(n, 1)[0], scratch(qg)
    call(lib.qmhd_ct_emf, C.byref(qg), order, flags(sides), G53, *[ptrs(x) for x in dev], C.c_void_p(ez.data_ptr()),
         C.c_void_p(sc.data_ptr()), None)
    m = flux_mask(nx, ny, ng)
    got, ref = to_host([ez])[0][m], want[m]
    assert np.isfinite(ref).all()
    assert np.abs(got - ref).sum() <= 1e-13 * max(np.abs(ref).sum(), 1e-3 * len(ref))
