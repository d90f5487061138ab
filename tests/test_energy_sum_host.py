"""The energy's three-term sum when a face state takes its normal field (en + v^2/2 -
bn^2/2, correctly rounded), built for the host from the kernels' own function: a sum
that it calls certain has the exact sum's bits, and it is certain wherever the sum is
not within its last error of a midpoint, so a nearly vanishing normal field does not
send a face to the general path."""
import ctypes as C
import subprocess
from fractions import Fraction

import numpy as np
import pytest

from host_kernels_ctypes import HOST_SO

N = 100_000


@pytest.fixture(scope="module")
def sums():
    subprocess.run(["make", "-C", str(HOST_SO.parents[1])], check=True, stdout=subprocess.DEVNULL)
    fn = C.CDLL(str(HOST_SO.with_name("libface_kernels.so"))).fk_sum_of_three
    fn.argtypes = [C.c_long] + [C.c_void_p] * 4

    def call(terms):
        terms = np.ascontiguousarray(terms)
        total, exact, sure = np.empty(len(terms)), np.empty(len(terms)), np.empty(len(terms), np.int32)
        fn(len(terms), terms.ctypes.data, total.ctypes.data, sure.ctypes.data, exact.ctypes.data)
        return total, sure != 0, exact

    return call


def terms_of(field, change, rng):
    v = field * rng.normal(size=N)
    bn = v * (1 + change * rng.normal(size=N))
    return np.column_stack([rng.uniform(0.1, 10, N), v * (0.5 * v), -(bn * (0.5 * bn))])


@pytest.mark.parametrize("field", [1.0, 1e-2, 1e-5, 1e-7, 1e-8, 1e-9, 1e-12, 1e-20, 1e-100, 1e-160])
@pytest.mark.parametrize("change", [1e-12, 1e-6, 1e-2, 1.0])
def test_the_sum_is_certain_and_exact(sums, field, change):
    t = terms_of(field, change, np.random.default_rng(1))
    total, sure, exact = sums(t)
    assert np.array_equal(total[sure], exact[sure])
    assert sure.mean() > 0.999
    for row, x in list(zip(t[sure], total[sure]))[:200]:
        assert float(sum(map(Fraction, row))) == x


def test_a_sum_next_to_a_midpoint_is_not_called_certain_on_the_wrong_side(sums):
    rng = np.random.default_rng(2)
    a = rng.uniform(1, 2, N)
    half = np.full(N, 2.0 ** -53)  # half a spacing in [1, 2)
    for small in (1e-40, 1e-33, 1e-30, 1e-25, 1e-20):
        t = np.column_stack([a, half, small * rng.normal(size=N)])
        for order in ([0, 1, 2], [0, 2, 1], [1, 0, 2]):
            total, sure, exact = sums(t[:, order])
            assert np.array_equal(total[sure], exact[sure])
            for row, x in list(zip(t, exact))[:50]:
                assert float(sum(map(Fraction, row))) == x


def test_nothing_that_is_not_finite_is_certain(sums):
    bad = [np.nan, np.inf, -np.inf]
    t = np.array([[b if k == m else 1.0 for m in range(3)] for b in bad for k in range(3)])
    assert not sums(t)[1].any()
