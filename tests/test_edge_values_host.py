"""The corner E_z's edge values (average -> edge interpolation), built for the host
from the kernels' own function, against the weighted sum in extended precision.

Bound, in roundings (2^-53) of the largest sample: one for the last addition, plus
what the pair sums round, each at twice its weight: 2 (139 + 29 + 3 + 113) / 840 =
0.68 for eight samples, 2 (8 + 1 + 7) / 60 = 0.54 for six; plus three times the
weights' share of the samples' spread for the differences and products."""
import ctypes as C
import subprocess

import numpy as np
import pytest

from host_kernels_ctypes import HOST_SO

WEIGHTS = {7: (np.array([-3, 29, -139, 533, 533, -139, 29, -3], np.longdouble), 840),
           5: (np.array([1, -8, 37, 37, -8, 1], np.longdouble), 60)}


@pytest.fixture(scope="module")
def edge_interp():
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    fn = C.CDLL(str(HOST_SO.with_name("libface_kernels.so"))).fk_edge_interp
    fn.argtypes = [C.c_int, C.c_long, C.c_void_p, C.c_void_p]

    def call(order, e):
        e = np.ascontiguousarray(e)
        out = np.empty(len(e))
        fn(order, len(e), e.ctypes.data, out.ctypes.data)
        return out

    return call


@pytest.mark.parametrize("order, sums", [(7, 0.68), (5, 0.54)])
@pytest.mark.parametrize("spread", [1e-2, 1e-5])
def test_a_smooth_value_rounds_once_at_its_size(edge_interp, order, sums, spread):
    w, scale = WEIGHTS[order]
    rng = np.random.default_rng(order)
    e = (1 + spread * rng.normal(size=(200_000, order + 1))) * rng.choice([-1, 1], (200_000, 1))
    exact = e.astype(np.longdouble) @ w / scale
    err = np.abs((edge_interp(order, e) - exact).astype(np.float64)) / np.abs(e).max(1)
    assert err.max() <= (1 + sums + 3 * 6 * spread) * 2.0 ** -53


@pytest.mark.parametrize("order", [5, 7])
def test_equal_samples_give_that_sample(edge_interp, order):
    v = np.random.default_rng(0).normal(size=1000) * 10.0 ** np.random.default_rng(1).integers(-200, 200, 1000)
    assert np.array_equal(edge_interp(order, np.repeat(v[:, None], order + 1, 1)), v)
