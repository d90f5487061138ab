"""The biorthogonality test of the wave basis, which shares products between the
two waves of a pair, decides as the test that forms every row and column by
itself: on states of all kinds, and on scales where about half fail it."""
import numpy as np
import pytest

from test_face_logic_host import _states, fk  # noqa: F401


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("kind", ["general", "no_transverse", "small_transverse", "small_normal", "umbilic", "planar",
                                  "cold", "at_rest", "scaled"])
def test_shared_products_decide_alike(fk, kind, fp32):  # noqa: F811
    rng = np.random.default_rng(7)
    n = 40000
    for gamma in (1.4, 5.0 / 3.0):
        s = _states("general" if kind == "scaled" else kind, n, gamma, rng)
        if kind == "scaled":
            q = 10.0 ** rng.uniform(-4, 4, (n, 1))  # rho x q, velocity / sqrt(q), pressure and field as they are
            s[:, :1] *= q
            s[:, 1:4] *= np.sqrt(q)
        out = np.zeros(n, dtype=np.int32)
        fk.fk_basis_decisions(fp32, n, s.ctypes.data, gamma, out.ctypes.data)
        np.testing.assert_array_equal(out & 4 != 0, out & 8 != 0)
        if kind == "scaled":
            assert 0.05 < np.mean(out & 4 != 0) < 0.95
