"""Calls of several host threads on one stream: every call gets its own
result, whatever the others start in between.
"""
import ctypes as C
import threading

import numpy as np
import pytest

import honei_amd as H
import oracle

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
@pytest.mark.parametrize("n", [1, 2048, 2049, 100003])
def test_sums_that_return(n, kind, dtype):
    """One work-group's sum and sums over partials; the results of the same
    calls one after another."""
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


def test_sums_left_on_the_device():
    """The same for sums that stay on the device, a defect's norm among them."""
    n, side, rounds = 60001, 257, 60
    rng = np.random.default_rng(5)
    xs = [H.DeviceArray.from_host(rng.standard_normal(n)) for _ in range(2)]
    D = H.DeviceEll.from_oracle(oracle.q1_matrix(side))
    x, b, r = (H.DeviceArray.from_host(rng.standard_normal(side * side)) for _ in range(3))

    def call(k, out, j):
        at = H._p(out.ptr + 8 * j)
        if k == 0:
            H.call("honei_hip_dot_product_dev", H.F64, at, xs[0].ptr, xs[1].ptr, n, None)
        elif k == 1:
            H.call("honei_hip_norm_l2_dev", H.F64, at, xs[1].ptr, n, None)
        else:
            H.call("honei_hip_defect_norm_smell_dv", D.vtype, b.ptr, r.ptr, D.Aj.ptr, D.Ax.ptr, D.Arl.ptr, x.ptr, D.rows,
                   D.ncpr, D.stride, D.threads, at, None)

    outs = [H.DeviceArray(rounds + 1, np.float64) for _ in range(3)]
    for k in range(3):
        call(k, outs[k], rounds)

    def work(k):
        for j in range(rounds):
            call(k, outs[k], j)

    assert not _run(3, work)
    H.call("honei_hip_synchronize", None)
    for k in range(3):
        got = outs[k].get()
        assert (got == got[rounds]).all(), k


def test_solves_and_sums():
    """CG and PCG-Jacobi solves (of more and more rows: the scratch grows), and
    sums beside them: the results of the same calls one after another."""
    n, sides = 50021, [33, 65, 129, 257]
    rng = np.random.default_rng(9)
    x = H.DeviceArray.from_host(rng.standard_normal(n))
    systems = []
    for side in sides:
        b = rng.standard_normal((side, side))
        b[0] = b[-1] = b[:, 0] = b[:, -1] = 0
        systems.append((H.DeviceEll.from_oracle(oracle.q1_matrix(side)), H.DeviceArray.from_host(b.ravel()),
                        H.DeviceArray.from_host(np.full(side * side, 0.375))))

    def solve(pcg, i):
        D, b, dinv = systems[i]
        u = H.DeviceArray.from_host(np.zeros(b.n))
        r = (H.pcg_jacobi(D, b, u, dinv, 400, 1e-9, check=False) if pcg else
             H.cg_solve(D, b, u, 400, 1e-9, check=False))
        return r, u.get().tobytes()

    sums = _reduce("dot", x, x)
    want = {(pcg, i): solve(pcg, i) for pcg in (0, 1) for i in range(len(sides))}
    bad = []

    def work(k):
        if k < 3:
            for i in range(len(sides)):
                if solve(k % 2, i) != want[k % 2, i]:
                    bad.append((k, i))
        else:
            for j in range(200):
                if _reduce("dot", x, x) != sums:
                    bad.append((k, j))

    assert not _run(5, work)
    assert not bad, bad[:5]
