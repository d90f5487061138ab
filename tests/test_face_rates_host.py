"""Signal speeds of faces whose pressure is within rounding of zero (the step
kernels' face functions built for the host): infinite where the reference's
pressure of a side is not positive, finite where it is, whatever the order of
rounding of the fast path.  An infinite speed stops a run."""
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
    L.fk_fluxes.argtypes = [C.c_int, C.c_int, C.c_int, C.c_long, C.c_void_p, C.c_int, C.c_double, C.c_void_p, C.c_void_p]
    return L


@pytest.mark.parametrize("order,width", [(1, 1), (2, 1), (5, 5), (7, 7)])
@pytest.mark.parametrize("d", [0, 1])
def test_rate_follows_the_reference_pressure(oracle, fk, order, width, d):
    rng = np.random.default_rng(order + 10 * d)
    n, gamma = 4000, 5 / 3
    rho, m, b = 10 ** rng.uniform(-2, 2, n), rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    en = 0.5 * (m ** 2).sum(1) / rho + 0.5 * (b ** 2).sum(1)
    en = en + rng.integers(-4, 5, n) * np.spacing(en)
    u = np.column_stack([rho, m, en, b])
    positive = np.array([oracle.pressure(x, gamma) > 0 for x in u])
    assert 0.3 < positive.mean() < 0.7
    # The same averages along the face line: every point has the averages' state.
    s = np.ascontiguousarray(np.repeat(np.concatenate([u, u], axis=1)[:, :, None], width, axis=2))
    flux, rate = np.zeros((n, 8)), np.zeros(n)
    fk.fk_fluxes(0, order, 0, n, s.ctypes.data, d, gamma, flux.ctypes.data, rate.ctypes.data)
    np.testing.assert_array_equal(np.isfinite(rate), positive)
