"""Dot products and sums around the size up to which one block takes them."""
import ctypes
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import alp_amd
    alp_amd.init(0)
    return alp_amd


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 8191, 8192, 8193, 16383, 16384, 16385])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_dot_and_sum(A, n, dtype):
    """n products and sums in FP64, each within 2^-53 of the terms' size (FP32
    products are exact); the start value is added once; repeats are identical."""
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal(n).astype(dtype), rng.standard_normal(n).astype(dtype)
    X, Y = A.Vector.from_numpy(x), A.Vector.from_numpy(y)
    prod = x.astype(np.float64) * y.astype(np.float64)
    bound = (n + 1) * 2.0 ** -53 * (np.abs(prod).sum() + 3.0)
    f = A.lib().alp_hip_dot_f64 if dtype == np.float64 else A.lib().alp_hip_dot_f32
    got = []
    for _ in range(2):
        z = ctypes.c_double(3.0)
        A.check(f(n, X.ptr, Y.ptr, ctypes.byref(z)), "dot")
        got.append(z.value)
    assert got[0] == got[1]
    assert abs(got[0] - (math.fsum(prod) + 3.0)) <= bound
    if dtype == np.float64:
        z = ctypes.c_double(-1.0)
        A.check(A.lib().alp_hip_sum_f64(n, X.ptr, ctypes.byref(z)), "sum")
        assert abs(z.value - (math.fsum(x) - 1.0)) <= (n + 1) * 2.0 ** -53 * (np.abs(x).sum() + 1.0)
