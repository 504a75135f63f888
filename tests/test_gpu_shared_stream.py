"""Calls of several host threads on one stream: every call gets its own
result, whatever the others start in between.
"""
import ctypes as C
import threading

import numpy as np
import pytest

import honei_amd as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _run(count, work):
    """work(k) on `count` threads that start together; their exceptions."""
    gate, errors = threading.Barrier(count), []

    def body(k):
        try:
            gate.wait()
            work(k)
        except Exception as e:   # noqa: BLE001 -- reported by the caller
            errors.append((k, e))

    threads = [threading.Thread(target=body, args=(k,)) for k in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    return errors


def _reduce(kind, x, y, stream=None):
    v = (C.c_double if x.dtype == np.float64 else C.c_float)()
    name = "double" if x.dtype == np.float64 else "float"
    if kind == "dot":
        H.call("honei_hip_dot_product_two_" + name, C.byref(v), x.ptr, y.ptr, x.n, stream)
    else:
        H.call("honei_hip_norm_l2_one_" + name, C.byref(v), x.ptr, x.n, stream)
    return v.value


def test_more_waiting_calls_than_kept_results():
    """100 calls started while the stream is still busy with earlier work, so
    that all of them wait for their results at the same time."""
    p = H._p()
    H.call("honei_hip_stream_create", C.byref(p))
    n, calls = 1500, 100
    ones = H.DeviceArray.from_host(np.ones(n))
    arrays = [H.DeviceArray.from_host(np.full(n, float(k + 1))) for k in range(calls)]
    busy = H.DeviceArray(1 << 26, np.float64)
    got = [None] * calls
    H.call("honei_hip_synchronize", None)
    for _ in range(1500):   # 0.8 TB of stores: some 150 ms
        H.call("honei_hip_fill", H.F64, busy.ptr, 1.0, busy.n, p.value)

    def work(k):
        got[k] = _reduce("dot", arrays[k], ones, p.value)

    assert not _run(calls, work)
    assert got == [n * (k + 1.0) for k in range(calls)]
    H.call("honei_hip_stream_destroy", p.value)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["dot", "norm"])
@pytest.mark.parametrize("n", [1, 2048])
def test_sums_that_return(n, kind, dtype):
    """Sums of one work-group; the results of the same calls one after another."""
    rng = np.random.default_rng(n)
    arrays = [H.DeviceArray.from_host(rng.standard_normal(n).astype(dtype)) for _ in range(6)]
    want = [_reduce(kind, a, arrays[0]) for a in arrays]
    bad = []

    def work(k):
        for _ in range(150):
            v = _reduce(kind, arrays[k], arrays[0])
            if v != want[k]:
                bad.append((k, v))

    assert not _run(6, work)
    assert not bad, (len(bad), bad[:4], want)
