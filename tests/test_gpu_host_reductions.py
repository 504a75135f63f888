"""Dot products and norms that return to the host: one work-group and several,
empty and special values, and calls from several threads at once.
"""
import ctypes
import math
import threading

import numpy as np
import pytest

import honei_amd as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _dot(x, y, n, dtype):
    v = (ctypes.c_double if dtype == np.float64 else ctypes.c_float)()
    H.call("honei_hip_dot_product_two_" + ("double" if dtype == np.float64 else "float"), ctypes.byref(v), x.ptr, y.ptr,
           n, None)
    return v.value


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [0, 1, 255, 2047, 2048, 2049, 4097, 100003])
def test_dot(n, dtype):
    rng = np.random.default_rng(n)
    x, y = (rng.standard_normal(max(n, 1)).astype(dtype) for _ in range(2))
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray.from_host(y)
    got = _dot(dx, dy, n, dtype)
    terms = [float(a) * float(b) for a, b in zip(x[:n], y[:n])]
    # sums in double: n roundings of partial sums below sum |terms|, and the result's own
    bound = n * 2.0 ** -53 * math.fsum(map(abs, terms)) + np.finfo(dtype).eps * abs(math.fsum(terms))
    assert abs(got - math.fsum(terms)) <= bound
    out = H.DeviceArray(1, np.float64)
    H.call("honei_hip_dot_product_dev", H.F64 if dtype == np.float64 else H.F32, out.ptr, dx.ptr, dy.ptr, n, None)
    assert got == dtype(out.get()[0])


@pytest.mark.parametrize("n", [5, 3000])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_special_values(n, value):
    x = np.ones(n)
    x[n // 2] = value
    d = H.DeviceArray.from_host(x)
    assert np.array_equal(_dot(d, d, n, np.float64), value, equal_nan=True)
    x[:] = -0.0
    assert _dot(H.DeviceArray.from_host(x), H.DeviceArray.from_host(np.ones(n)), n, np.float64) == 0.0


def test_threads():
    """More calls than the results kept at a time, from several threads."""
    n, bad = 1500, []
    arrays = [H.DeviceArray.from_host(np.full(n, float(k + 1))) for k in range(4)]

    def work(k):
        for _ in range(100):
            if _dot(arrays[k], arrays[0], n, np.float64) != n * (k + 1.0):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("partials", [1, 1024, 1025, 4096, 4097, 8193])
def test_sums_of_partials(partials):
    """A defect's norm from one partial per 256 rows, on both sides of the rule
    for loading them one by one or eight at a time: integers, so exact."""
    n = 256 * (partials - 1) + 17
    stride = 32 * ((n + 31) // 32)
    b = np.random.default_rng(partials).integers(-8, 9, n).astype(np.float64)
    D = H.DeviceEll(n, n, stride, 1, 1, np.zeros(stride, np.uint64), np.zeros(stride), np.zeros(n, np.uint64), H.F64)
    db, x, r, out = (H.DeviceArray.from_host(b), H.DeviceArray.from_host(b), H.DeviceArray(n, np.float64),
                     H.DeviceArray(1, np.float64))
    D.defect_norm(r, db, x, out)
    assert out.get()[0] == (b * b).sum()
    assert np.array_equal(r.get(), b)
