"""The step kernels' face solver, FP32 reconstruction and cell E_z quadrature,
built for the host from the kernels' own functions, against the oracle.

Bound: 450 epsilon of the arithmetic in relative L1 (1e-13 in FP64, the bound of
every launch; 5.4e-5 in FP32), each flux component against its face's largest."""
import ctypes as C
import subprocess

import numpy as np
import pytest

from host_kernels_ctypes import HOST_SO

FACES_SO = HOST_SO.with_name("libface_kernels.so")
G53 = 5.0 / 3.0
BOUND = {0: 450 * np.finfo(np.float64).eps, 1: 450 * np.finfo(np.float32).eps}


@pytest.fixture(scope="module")
def fk():
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    L = C.CDLL(str(FACES_SO))
    P = C.c_void_p
    L.fk_fluxes.argtypes = [C.c_int, C.c_int, C.c_int, C.c_long, P, C.c_int, C.c_double, P, P]
    for f in (L.fk_mp_faces, L.fk_mp_faces_fp32):
        f.argtypes = [C.c_int, C.c_long, P, P, C.c_double, P, P]
    L.fk_cell_ez.argtypes = [C.c_int, C.c_long, P, P, P]
    return L


def cons(rho, p, v, b):
    return np.column_stack([rho, *(rho * q for q in v), p / (G53 - 1) + 0.5 * rho * sum(q * q for q in v) +
                            0.5 * sum(q * q for q in b), *b])


def pair(kind, n, rng):
    normal = lambda: [rng.normal(size=n) for _ in range(3)]
    (rl, rr), (pl, pr) = 10 ** rng.uniform(-1, 1, (2, n)), 10 ** rng.uniform(-1, 1, (2, n))
    vl, vr, bl, br = normal(), normal(), normal(), normal()
    br[0] = bl[0]
    if kind == "equal":
        return (cons(rl, pl, vl, bl),) * 2
    if kind == "no_normal":
        bl[0] = br[0] = np.zeros(n)
    elif kind == "tiny_normal":
        bl[0] = br[0] = 1e-9 * bl[0]
    elif kind == "no_transverse":
        bl[1:] = br[1:] = [np.zeros(n)] * 2
    elif kind == "supersonic":
        vl[0], vr[0] = vl[0] + 30, vr[0] + 30
    elif kind == "separating":
        vl[0], vr[0] = vl[0] - 3, vr[0] + 3
    elif kind == "contact":
        vr, pr, br = vl, pl, bl
    elif kind == "split_normal":
        br[0] = bl[0] + 0.1
    return cons(rl, pl, vl, bl), cons(rr, pr, vr, br)


SWAP = [0, 2, 1, 3, 4, 6, 5, 7]


def fluxes(fk, fp32, order, lf, left, right, d=0):
    s = np.ascontiguousarray(np.concatenate([left, right], axis=1)[:, :, None])
    flux, rate = np.zeros((len(left), 8)), np.zeros(len(left))
    fk.fk_fluxes(fp32, order, lf, len(left), s.ctypes.data, d, G53, flux.ctypes.data, rate.ctypes.data)
    return flux, rate


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("kind", ["general", "equal", "no_normal", "tiny_normal", "no_transverse", "supersonic",
                                  "separating", "contact", "split_normal"])
def test_flux_of_two_states(oracle, fk, kind, fp32):
    rng = np.random.default_rng(len(kind))
    left, right = pair(kind, 2000, rng)
    if fp32:
        left, right = left.astype(np.float32).astype(float), right.astype(np.float32).astype(float)
    want = np.array([oracle.hlld_flux_x(a, b, G53) for a, b in zip(left, right)])
    got, rate = fluxes(fk, fp32, 2, 0, left, right)
    scale = np.abs(want).max(axis=1, keepdims=True)
    assert np.isfinite(rate).all()
    assert (np.abs(got - want) / scale).mean(axis=0).max() <= BOUND[fp32]
    turned, rate_y = fluxes(fk, fp32, 2, 0, left[:, SWAP], right[:, SWAP], 1)
    np.testing.assert_array_equal(turned[:, SWAP], got)
    np.testing.assert_array_equal(rate_y, rate)
    want = np.array([oracle.lf_flux_x(a, b, G53) for a, b in zip(left, right)])
    got, _ = fluxes(fk, fp32, 1, 1, left, right)
    assert (np.abs(got - want) / np.abs(want).max(axis=1, keepdims=True)).mean(axis=0).max() <= BOUND[fp32]


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("comp", range(5))
def test_flux_beside_a_nan(oracle, fk, comp, side):
    """A NaN in one state leaves the flux finite where the reference's choices
    drop it, and nowhere else; the signal speed is infinite."""
    states = [q.copy() for q in pair("general", 500, np.random.default_rng(2))]
    states[side][:, comp] = np.nan
    want = np.array([oracle.hlld_flux_x(a, b, G53) for a, b in zip(*states)])
    got, rate = fluxes(fk, 0, 2, 0, *states)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    f = np.isfinite(want)
    assert np.all(np.abs(got[f] - want[f]) <= 1e-11 * np.maximum(1, np.abs(want[f])))
    assert np.isposinf(rate).all()


def smooth_planes(nx, ny, ng, rng):
    y, x = np.mgrid[0:ny + 2 * ng, 0:nx + 2 * ng]
    w = lambda a, b: np.sin(2 * np.pi * (x / 17 + a)) * np.cos(2 * np.pi * (y / 13 + b)) + 0.05 * rng.normal(size=x.shape)
    rho, p = 1 + 0.2 * w(0.1, 0.2), 1 + 0.2 * w(0.3, 0.7)
    v, b = [0.3 * w(k, 0.3) for k in (0.2, 0.6, 0.8)], [0.5 + 0.2 * w(k, 0.6) for k in (0.5, 0.4, 0.9)]
    return [np.ascontiguousarray(q).ravel() for q in cons(rho.ravel(), p.ravel(), [q.ravel() for q in v],
                                                          [q.ravel() for q in b]).T]


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("order,ng", [(5, 3), (7, 4)])
@pytest.mark.parametrize("d", [0, 1])
def test_flux_over_nodes(oracle, fk, d, order, ng, fp32):
    nx, ny, h = 21, 19, 2 if order == 5 else 3
    rng = np.random.default_rng(order + d)
    g = oracle.grid(nx, ny, ng)
    iface = smooth_planes(nx, ny, ng, rng) + smooth_planes(nx, ny, ng, rng)
    iface[8 + 5 + d] = iface[5 + d]
    if fp32:
        iface = [q.astype(np.float32).astype(float) for q in iface]
    want = [np.zeros_like(iface[0]) for _ in range(8)]
    oracle.face_flux(g, d, order, 0, (1, 1, 1, 1), G53, iface, want)
    pitch = nx + 2 * ng
    k = np.array([(i + ng) + pitch * (j + ng) for j in range(ny) for i in range(nx)])
    step = pitch if d == 0 else 1
    s = np.ascontiguousarray(np.array([[iface[c][k + m * step] for m in range(-h, h + 1)] for c in range(16)])
                             .transpose(2, 0, 1))
    flux, rate = np.zeros((len(k), 8)), np.zeros(len(k))
    fk.fk_fluxes(fp32, order, 0, len(k), s.ctypes.data, d, G53, flux.ctypes.data, rate.ctypes.data)
    ref = np.array([q[k] for q in want]).T
    assert (np.abs(flux - ref) / np.abs(ref).max(axis=1, keepdims=True)).mean(axis=0).max() <= BOUND[fp32]


@pytest.mark.parametrize("order,ng", [(5, 3), (7, 4)])
def test_reconstruction_in_fp32(oracle, fk, order, ng):
    """FP32 faces follow FP64 ones of the same (FP32) cells, but for decisions
    near their thresholds: the median and the mean are rounding."""
    h = order // 2
    rng = np.random.default_rng(order)
    n = 4000
    q = np.arange(order + 1)[None, :]
    wave = lambda: 0.1 * np.sin(0.3 * q + 6 * rng.random((n, 1))) + 0.01 * rng.normal(size=(n, order + 1))
    rho, p, v, b = 1 + wave(), 1 + wave(), [wave() for _ in range(3)], [0.5 + wave() for _ in range(3)]
    cells = cons(rho.ravel(), p.ravel(), [x.ravel() for x in v], [x.ravel() for x in b])
    cells = np.ascontiguousarray(cells.reshape(n, order + 1, 8).transpose(0, 2, 1).astype(np.float32).astype(float))
    bn = np.ascontiguousarray(cells[:, 5, h])
    out = []
    for f in (fk.fk_mp_faces, fk.fk_mp_faces_fp32):
        o, settled = np.zeros((n, 16)), np.zeros(n, dtype=np.int32)
        f(order, n, cells.ctypes.data, bn.ctypes.data, G53, o.ctypes.data, settled.ctypes.data)
        assert settled.mean() > 0.99
        out.append((o, settled.astype(bool)))
    both = out[0][1] & out[1][1]
    error = np.abs(out[0][0] - out[1][0])[both]
    assert np.median(error) <= 4 * np.finfo(np.float32).eps
    assert error.mean() <= BOUND[1]


@pytest.mark.parametrize("order,ng", [(5, 3), (7, 4)])
def test_cell_ez_quadrature(oracle, fk, order, ng):
    nx, ny, h = 15, 14, order // 2
    rng = np.random.default_rng(order)
    g = oracle.grid(nx, ny, ng)
    u = smooth_planes(nx, ny, ng, rng)
    flags = (1, 1, 1, 1)
    faces = [[np.zeros_like(u[0]) for _ in range(16)] for _ in range(2)]
    for d in (0, 1):
        oracle.reconstruct(g, d, order, flags, G53, u, faces[d])
    want = oracle.ct_emf(g, order, 0, flags, G53, u, *faces)["cell_ez"]
    pitch = nx + 2 * ng
    planes = [p.copy() for p in u]
    for j in range(-ng, ny + ng):
        for i in range(-ng, nx + ng):
            at = (i + ng) + pitch * (j + ng)
            planes[5][at], planes[6][at] = oracle.cell_bx(g, u[5], i, j, 0), oracle.cell_by(g, u[6], i, j, 0)
    k = np.array([(i + ng) + pitch * (j + ng) for j in range(ny) for i in range(nx)])
    s = np.ascontiguousarray(np.array([[[p[k + y * pitch + x] for x in range(-h, h + 1)] for y in range(-h, h + 1)]
                                       for p in planes]).transpose(3, 0, 1, 2))
    ez, ok = np.zeros(len(k)), np.zeros(len(k), dtype=np.int32)
    fk.fk_cell_ez(order, len(k), s.ctypes.data, ez.ctypes.data, ok.ctypes.data)
    assert ok.all()
    assert np.abs(ez - want[k]).sum() <= BOUND[0] * np.abs(want[k]).sum()
