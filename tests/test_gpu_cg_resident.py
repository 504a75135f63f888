"""CG and PCG-Jacobi in resident launches against the launch-by-launch
iteration: a matrix stored with one more (empty) slot per row than the
resident form takes has the same rows and goes launch by launch, so x, the
iteration count and the final defect have to be the same bits.
"""
import threading

import numpy as np
import pytest

import honei_amd as H
from tests.patterns import uniform_pm1

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _ell(cols, vals, arl, width, vtype):
    """DeviceEll (threads 1) of [row][k] entries stored `width` slots wide."""
    n, k = cols.shape
    stride = 32 * ((n + 31) // 32)
    Aj = np.zeros((width, stride), np.uint64)
    Ax = np.zeros((width, stride), np.float64 if vtype == H.F64 else np.float32)
    Aj[:k, :n], Ax[:k, :n] = cols.T, vals.T
    return H.DeviceEll(n, n, stride, width, 1, Aj.ravel(), Ax.ravel(), arl, vtype)


def _tridiagonal(n, shift):
    """Rows (-1, 2 + shift, -1), entries ascending, two or fewer at the ends."""
    r = np.arange(n)
    cols = np.stack([r - 1, r, r + 1], 1)
    vals = np.tile(np.array([-1.0, 2.0 + shift, -1.0]), (n, 1))
    arl = np.full(n, 3)
    cols[0], vals[0] = [0, 1, 0], [2.0 + shift, -1.0, 0.0]
    arl[0] = 2
    arl[n - 1] -= 1
    if n == 1:
        arl[0] = 1
    cols = np.where(np.arange(3)[None, :] < arl[:, None], cols, 0)
    vals = np.where(np.arange(3)[None, :] < arl[:, None], vals, 0.0)
    return cols, vals, arl


def _grid(side):
    """Nine-point operator, identity boundary rows (widths 1 and 9)."""
    n = side * side
    r = np.arange(n)
    edge = (r < side) | (r >= n - side) | (r % side == 0) | (r % side == side - 1)
    offs = np.array([-side - 1, -side, -side + 1, -1, 0, 1, side - 1, side, side + 1])
    cols = np.where(edge[:, None], 0, r[:, None] + offs)
    vals = np.where(edge[:, None], 0.0, np.where(offs == 0, 8 / 3, -1 / 3)[None, :])
    cols[edge, 0], vals[edge, 0] = r[edge], 1.0
    return cols, vals, np.where(edge, 1, 9)


def _solve(D, b, dinv, eps, max_iters, stream=None):
    db, dx = H.DeviceArray.from_host(b), H.DeviceArray.from_host(np.zeros_like(b))
    if dinv is None:
        used, fd = H.cg_solve(D, db, dx, max_iters, eps, stream=stream, check=False)
    else:
        used, fd = H.pcg_jacobi(D, db, dx, H.DeviceArray.from_host(dinv), max_iters, eps, stream=stream, check=False)
    return dx.get(), used, fd


def _same(system, vtype, pcg, eps, max_iters=20000):
    cols, vals, arl = system
    dt = np.float64 if vtype == H.F64 else np.float32
    b = uniform_pm1(7, arl.size).astype(dt)
    b[arl == 1] = 0
    dinv = None
    if pcg:
        diag = np.where((cols == np.arange(arl.size)[:, None]) & (vals != 0), vals, 0.0).sum(1)
        dinv = (uniform_pm1(8, arl.size) * 0.25 + 1.0).astype(dt) / diag.astype(dt)
    x1, u1, f1 = _solve(_ell(cols, vals, arl, 9, vtype), b, dinv, eps, max_iters)
    x2, u2, f2 = _solve(_ell(cols, vals, arl, 10, vtype), b, dinv, eps, max_iters)
    assert u1 == u2 and f1 == f2, (u1, u2, f1, f2)
    assert np.array_equal(x1.view(np.uint8), x2.view(np.uint8))
    return u1


# rows around a partial (256), a group (2048), the split of groups (65,536)
# and the largest that fits (2048 partials)
ROWS = [1, 2, 63, 255, 256, 257, 2047, 2049, 65535, 65537, 524288, 524289]


@pytest.mark.parametrize("pcg", [False, True])
@pytest.mark.parametrize("n", ROWS)
def test_rows(n, pcg):
    _same(_tridiagonal(n, 0.05), H.F64, pcg, 1e-10)


@pytest.mark.parametrize("vtype", [H.F32, H.F64, H.BF16])
@pytest.mark.parametrize("pcg", [False, True])
@pytest.mark.parametrize("side", [3, 33, 255, 257])
def test_grids(side, pcg, vtype):
    _same(_grid(side), vtype, pcg, 1e-9 if vtype == H.F64 else 1e-5, 3000)


@pytest.mark.parametrize("max_iters", [1, 2, 4095, 4096, 4097])
def test_iteration_limits(max_iters):
    """A limit inside, at and beyond one launch; the system needs more."""
    assert _same(_tridiagonal(12000, 0.0), H.F64, False, 1e-14, max_iters) == max_iters


def test_threads_and_streams():
    """Solves from several threads, each on its own stream, at once: the
    results of the same solves one after another."""
    systems = [(_grid(65), 1e-9), (_tridiagonal(70001, 0.05), 1e-10), (_grid(129), 1e-9), (_tridiagonal(300000, 0.1), 1e-9)]
    mats = [_ell(c, v, a, 9, H.F64) for (c, v, a), _ in systems]
    bs = []
    for (_, _, a), _ in systems:
        b = uniform_pm1(9, a.size)
        b[a == 1] = 0
        bs.append(b)
    want = [_solve(D, b, None, eps, 20000) for D, b, (_, eps) in zip(mats, bs, systems)]
    got, errors = [None] * 4, []

    def work(i):
        try:
            p = H._p()
            H.call("honei_hip_stream_create", H.C.byref(p))
            for _ in range(3):
                got[i] = _solve(mats[i], bs[i], None, systems[i][1], 20000, stream=p.value)
        except Exception as e:   # noqa: BLE001 -- reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errors, errors
    for (x1, u1, f1), (x2, u2, f2) in zip(want, got):
        assert u1 == u2 and f1 == f2 and np.array_equal(x1.view(np.uint8), x2.view(np.uint8))


@pytest.mark.parametrize("launch,max_iters,eps", [(0, 300, 1e-9), (1, 4500, 0.0)])
@pytest.mark.parametrize("pcg", [False, True])
@pytest.mark.parametrize("side,vtype", [(33, H.F64), (129, H.F32), (259, H.F64), (515, H.BF16)])
def test_given_up(side, vtype, pcg, launch, max_iters, eps):
    """A resident launch whose work-groups give up waiting -- the first, or one
    that continues from another's state -- leaves the launch-by-launch result.
    Sides: four, two and one work-groups per group of rows."""
    H.call("honei_hip_resident_give_up", launch)
    try:
        used = _same(_grid(side), vtype, pcg, eps, max_iters)
    finally:
        H.call("honei_hip_resident_give_up", -1)
    assert launch == 0 or used == max_iters


@pytest.mark.parametrize("max_iters", [1, 2, 3])
@pytest.mark.parametrize("pcg", [False, True])
@pytest.mark.parametrize("side,vtype", [(65, H.F32), (515, H.F64), (515, H.F32)])
def test_few_iterations(side, vtype, pcg, max_iters):
    """On both sides of the iteration count from which solves stay resident."""
    assert _same(_grid(side), vtype, pcg, 1e-9, max_iters) == max_iters
