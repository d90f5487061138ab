"""The MP5/MP7 face functions of the kernels, built for the host, against the
general path: the oracle's reconstruction on whole grids and its 1024-epsilon
decision state by state.

The decisions must agree exactly wherever the fast path takes one.  A settled
face is held to 1e-13 of max(1, |value|), as the general path's faces are: its
closed forms run where at most 2^10 separates the wave weights and the states
below are of order one."""
import ctypes as C
import subprocess

import numpy as np
import pytest

from host_kernels_ctypes import HOST_SO
from oracle_ctypes import ic_spec

FACES_SO = HOST_SO.with_name("libface_kernels.so")


@pytest.fixture(scope="module")
def fk():
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    L = C.CDLL(str(FACES_SO))
    L.fk_basis_decisions.argtypes = [C.c_int, C.c_long, C.c_void_p, C.c_double, C.c_void_p]
    L.fk_mp_faces.argtypes = [C.c_int, C.c_long, C.c_void_p, C.c_void_p, C.c_double, C.c_void_p, C.c_void_p]
    return L


def _states(kind, n, gamma, rng):
    rho, p = 10.0 ** rng.uniform(-2, 2, n), 10.0 ** rng.uniform(-3, 3, n)
    a = np.sqrt(gamma * p / rho)[:, None]
    v = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-2, 1, (n, 1)) * a
    b = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-2, 1, (n, 1)) * a * np.sqrt(rho)[:, None]
    if kind == "no_transverse":
        b[:, 1:] = 0.0
    elif kind == "small_transverse":
        b[:, 1:] *= 10.0 ** rng.uniform(-16, 0, (n, 1))
    elif kind == "small_normal":
        b[:, 0] *= 10.0 ** rng.uniform(-12, 0, n)
    elif kind == "umbilic":  # a close to the normal Alfven speed, little transverse field
        b[:, 0] = np.sqrt(rho) * a[:, 0] * (1 + rng.normal(size=n) * 10.0 ** rng.uniform(-12, 0, n))
        b[:, 1:] = rng.normal(size=(n, 2)) * b[:, :1] * 10.0 ** rng.uniform(-10, 0, (n, 1))
    elif kind == "planar":
        v[:, 2] = b[:, 2] = 0.0
    elif kind == "cold":
        p *= 10.0 ** rng.uniform(-12, 0, n)
    elif kind == "at_rest":
        v[:] = 0.0
    en = p / (gamma - 1) + 0.5 * rho * (v ** 2).sum(1) + 0.5 * (b ** 2).sum(1)
    return np.ascontiguousarray(np.column_stack([rho, rho[:, None] * v, en, b]))


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("kind", ["general", "no_transverse", "small_transverse", "small_normal", "umbilic", "planar",
                                  "cold", "at_rest"])
def test_basis_taken_as_usable_is_usable(fk, kind, fp32):
    rng = np.random.default_rng(11)
    n = 40000
    for gamma in (1.4, 5.0 / 3.0, 2.0):
        s = _states(kind, n, gamma, rng)
        out = np.zeros(n, dtype=np.int32)
        fk.fk_basis_decisions(fp32, n, s.ctypes.data, gamma, out.ctypes.data)
        assert not np.any((out & 1).astype(bool) & ~(out & 2).astype(bool))
        assert not np.any((out & 2).astype(bool) & ~(out & 4).astype(bool)), (kind, gamma)
        if kind == "general":
            assert np.mean(out & 1) > 0.2  # the fast path is exercised


@pytest.mark.parametrize("order", [5, 7])
@pytest.mark.parametrize("kind", ["orszag_tang", "rotor", "brio_wu", "noise"])
def test_settled_faces_match_oracle(oracle, fk, kind, order):
    nx, ny, ng, gamma = 21, 18, 4, 1.4
    g = oracle.grid(nx, ny, ng)
    F = (1, 1, 1, 1) if kind in ("rotor", "brio_wu") else (0, 0, 0, 0)
    kw = dict(orszag_tang=dict(b_uniform=[1 / np.sqrt(4 * np.pi), 0, 0], ot_rho=25 / (36 * np.pi),
                               ot_p=5 / (12 * np.pi), noise_amplitude=1e-3, noise_seed=3),
              rotor=dict(center=[0.5, 0.5], b_uniform=[5 / np.sqrt(4 * np.pi), 0, 0], p_ambient=1.0),
              brio_wu=dict(left=[1, 1, 0, 0, 0, 0.75, 1, 0], right=[0.125, 0.1, 0, 0, 0, 0.75, -1, 0]))
    if kind == "noise":
        rng = np.random.default_rng(5)
        n = (nx + 2 * ng) * (ny + 2 * ng)
        u = [1 + 0.1 * rng.random(n)] + [0.2 * rng.normal(size=n) for _ in range(3)] + [3 + rng.random(n)] + \
            [0.4 * rng.normal(size=n) for _ in range(3)]
    else:
        st, u = oracle.seed(g, ic_spec(kind, gamma, **kw[kind]))
        assert st == 0
    oracle.fill_ghosts(g, F, F, u)
    pitch = nx + 2 * ng
    H = (order - 1) // 2
    at = lambda i, j: (i + ng) + pitch * (j + ng)
    bxc, byc = np.zeros_like(u[0]), np.zeros_like(u[0])
    for j in range(-ng, ny + ng):
        for i in range(-ng, nx + ng):
            bxc[at(i, j)] = oracle.cell_bx(g, u[5], i, j, 0)
            byc[at(i, j)] = oracle.cell_by(g, u[6], i, j, 0)
    planes = [u[0], u[1], u[2], u[3], u[4], bxc, byc, u[7]]
    frame = {0: [0, 1, 2, 3, 4, 5, 6, 7], 1: [0, 2, 1, 3, 4, 6, 5, 7]}
    taken = 0
    for d in (0, 1):
        ref = [np.zeros_like(u[0]) for _ in range(16)]
        oracle.reconstruct(g, d, order, F, gamma, u, ref)
        k = np.array([at(i, j) for j in range(ny + d) for i in range(nx + 1 - d)])
        step = 1 if d == 0 else pitch
        cells = np.array([[planes[c][k + (q - H - 1) * step] for q in range(order + 1)] for c in frame[d]])
        cells = np.ascontiguousarray(cells.transpose(2, 0, 1))
        bn = np.ascontiguousarray(u[5 + d][k])
        out, settled = np.zeros((len(k), 16)), np.zeros(len(k), dtype=np.int32)
        fk.fk_mp_faces(order, len(k), cells.ctypes.data, bn.ctypes.data, gamma, out.ctypes.data, settled.ctypes.data)
        take = settled.astype(bool)
        taken += take.sum()
        for side in (0, 8):
            for c in range(8):
                want = ref[side + frame[d][c]][k][take]
                assert np.all(np.abs(out[take, side + c] - want) <= 1e-13 * np.maximum(1.0, np.abs(want))), (d, side + c)
    assert taken > nx * ny
