"""The face solver's device root and reciprocals against exact values.

sqrt_pos refines the hardware's reciprocal root once more with the rounded root,
so its second output is within the root's error (one half ulp, 2^-53 relative at
most in FP64, and what the last correction leaves, far below) and its own last
rounding of 1 / (2 sqrt(x)): under 2 epsilon (2^-52 in FP64, 2^-23 in FP32).
The root and the reciprocal are bounded by one epsilon."""
import ctypes as C
import pathlib

import numpy as np
import pytest

from gpu_helpers import torch_cuda

pytestmark = pytest.mark.gpu

SO = pathlib.Path(__file__).resolve().parent / "host_kernels" / "_build" / "libdevice_math.so"


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("span", [1, 30, 120, 400])
def test_roots_and_reciprocals(fp32, span):
    torch = torch_cuda()
    lib = C.CDLL(str(SO))
    lib.dm_roots.argtypes = [C.c_int, C.c_long] + [C.c_void_p] * 4
    t = np.float32 if fp32 else np.float64
    span = min(span, 60) if fp32 else span
    n = 1 << 18
    rng = np.random.default_rng(span)
    x = (rng.uniform(1, 2, n) * 2.0 ** rng.integers(-span, span, n)).astype(t)
    dev = torch.from_numpy(x).cuda()
    out = [torch.empty_like(dev) for _ in range(3)]
    torch.cuda.synchronize()
    assert lib.dm_roots(fp32, n, dev.data_ptr(), *[o.data_ptr() for o in out]) == 0
    root, half_inv, inv = [o.cpu().numpy().astype(np.longdouble) for o in out]
    q = x.astype(np.longdouble)
    eps = np.finfo(t).eps
    errors = [np.abs(a / b - 1).max() / eps for a, b in ((root, np.sqrt(q)), (half_inv, 0.5 / np.sqrt(q)), (inv, 1 / q))]
    print(f"{t.__name__} 2^+-{span}: root {errors[0]:.2f}, half inverse {errors[1]:.2f}, reciprocal {errors[2]:.2f} eps")
    assert errors[0] <= 1 and errors[1] <= 2 and errors[2] <= 1, errors
