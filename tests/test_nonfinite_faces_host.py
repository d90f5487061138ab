"""A value that is not finite anywhere in a face's stencil leaves the face to the
general path (the kernels' face function built for the host): its limiters are
made of minima and maxima, which drop a NaN, so a damaged cell must not come out
as a finite state."""
import ctypes as C
import subprocess

import numpy as np
import pytest

from host_kernels_ctypes import HOST_SO

FACES_SO = HOST_SO.with_name("libface_kernels.so")


@pytest.fixture(scope="module")
def fk():
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    L = C.CDLL(str(FACES_SO))
    L.fk_mp_faces.argtypes = [C.c_int, C.c_long, C.c_void_p, C.c_void_p, C.c_double, C.c_void_p, C.c_void_p]
    return L


def stencils(order, n, rough, rng):
    """(n, 8, order + 1) stencils of states of order one: smooth ones keep the
    unlimited value, rough ones take the limiters."""
    q = np.arange(order + 1)[None, :]
    wave = lambda a: 0.1 * np.sin(0.3 * q + 6 * rng.random((n, 1))) * a + rough * rng.normal(size=(n, order + 1))
    rho, p = 1 + wave(1), 1 + wave(1)
    v = [wave(1) for _ in range(3)]
    b = [0.5 + wave(0), 0.4 + wave(1), 0.3 + wave(1)]
    en = p / (5 / 3 - 1) + 0.5 * rho * sum(x * x for x in v) + 0.5 * sum(x * x for x in b)
    return np.ascontiguousarray(np.stack([rho, *(rho * x for x in v), en, *b], axis=1))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("rough", [0.0, 0.05])
@pytest.mark.parametrize("order", [5, 7])
def test_no_face_settles_beside_a_value_that_is_not_finite(fk, order, rough, bad):
    rng = np.random.default_rng(3)
    n = 64
    for cell in range(order + 1):
        for comp in range(8):
            # The normal field enters with the face's two own cells only.
            if comp == 5 and cell not in (order // 2, order // 2 + 1):
                continue
            cells = stencils(order, n, rough, rng)
            bn = np.ascontiguousarray(0.5 * (cells[:, 5, order // 2] + cells[:, 5, order // 2 + 1]))
            out, settled = np.zeros((n, 16)), np.zeros(n, dtype=np.int32)
            fk.fk_mp_faces(order, n, cells.ctypes.data, bn.ctypes.data, 5 / 3, out.ctypes.data, settled.ctypes.data)
            assert settled.mean() > 0.9  # without it they do
            cells[:, comp, cell] = bad
            fk.fk_mp_faces(order, n, cells.ctypes.data, bn.ctypes.data, 5 / 3, out.ctypes.data, settled.ctypes.data)
            assert not settled.any(), (comp, cell, int(settled.sum()))
