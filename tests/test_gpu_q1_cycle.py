"""Multigrid on device-assembled Q1 hierarchies: the matrix-free cycle and
outer iteration against the stored-matrix launches.

Setting the outer system of a built hierarchy (here to the very operator it
has) makes the solver assume no structure, so the same solve then runs level
by level on the stored matrices; solutions, counts and defects have to be the
same bits.
"""
import numpy as np
import pytest

import honei_amd as H
import oracle
from tests.patterns import lognormal_cells, poisson_system_seeds, uniform_pm1

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _operator(side, dk):
    n = side * side
    stride = 32 * ((n + 31) // 32)
    Aj, Ax, Arl = H.DeviceArray(9 * stride, np.int32), H.DeviceArray(9 * stride, np.float64), H.DeviceArray(n, np.uint32)
    H.call("honei_hip_q1_assemble", H.F64, side, Aj.ptr, Ax.ptr, Arl.ptr, stride, None if dk is None else dk.ptr, None,
           0.0, 1, None)
    return oracle.Ell(n, n, stride, 9, 1, Aj.get().astype(np.uint64), Ax.get(), Arl.get().astype(np.uint64))


def _both(level, inner, coeff, solve, **cfg):
    """(Q1 path, stored-matrix path) results of solve(mg, b, x)."""
    side = 2 ** level + 1
    cs, bs = poisson_system_seeds(77, level)
    dk = H.DeviceArray.from_host(lognormal_cells(cs, (side - 1) ** 2), np.float64) if coeff else None
    b = uniform_pm1(bs, side * side)
    out = []
    for stored in (False, True):
        mg = H.Multigrid(inner, 1, level)
        mg.configure(H.mg_config(**cfg))
        if coeff:
            mg.build_q1_coeff(dk, 0.8, 1)
        else:
            mg.build_q1(0.7)
        if stored:
            mg.set_outer(_operator(side, dk))
        db, dx = H.DeviceArray.from_host(b), H.DeviceArray(side * side, np.float64)
        for _ in range(2):   # a second solve on the same handle
            dx.zero()
            r = solve(mg, db, dx)
        out.append((r, dx.get()))
    (ra, xa), (rb, xb) = out
    assert ra == rb, (ra, rb)
    assert np.array_equal(xa, xb)
    assert np.isfinite(xa).all() and xa.any()


# coarse launch alone (2..6), its top and one / two paired levels above it
# (FP64: from 6), tall tiles and the fused direction pass (10)
LEVELS = [2, 3, 4, 5, 6, 7, 8, 10]


@pytest.mark.parametrize("inner", [H.F32, H.BF16, H.F64])
@pytest.mark.parametrize("coeff", [False, True])
@pytest.mark.parametrize("level", LEVELS)
def test_pcg(level, coeff, inner):
    _both(level, inner, coeff, lambda mg, b, x: mg.solve_pcg(b, x, check=False), tolerance=1e-9, max_outer=60)


@pytest.mark.parametrize("inner", [H.F32, H.BF16])
@pytest.mark.parametrize("coeff", [False, True])
@pytest.mark.parametrize("level", LEVELS)
def test_mixed_one_cycle(level, coeff, inner):
    _both(level, inner, coeff, lambda mg, b, x: mg.solve_mixed(b, x, check=False), n_max_iter=1, tolerance=1e-9,
          initial_zero=True, zero_inner_start=True, max_outer=25)


@pytest.mark.parametrize("level", [4, 7, 9])
def test_mixed_inner_cycles(level):
    """Several cycles per outer step from the carried-over start vector."""
    _both(level, H.F32, False, lambda mg, b, x: mg.solve_mixed(b, x, check=False), n_max_iter=4, tolerance=1e-9)


@pytest.mark.parametrize("level", [4, 6, 8])
def test_fixed(level):
    _both(level, H.F64, True, lambda mg, b, x: mg.solve_fixed(b, x), n_max_iter=6, tolerance=1e-12)


@pytest.mark.parametrize("cap", [1, 3, 4, 5])
def test_iteration_caps(cap):
    """The cap inside, at and beyond the first chunk of enqueued iterations."""
    _both(7, H.F32, True, lambda mg, b, x: mg.solve_pcg(b, x, check=False), tolerance=1e-14, max_outer=cap)
    _both(7, H.F32, False, lambda mg, b, x: mg.solve_mixed(b, x, check=False), n_max_iter=1, tolerance=1e-14,
          initial_zero=True, zero_inner_start=True, max_outer=cap)


@pytest.mark.parametrize("b", ["zero", "nan"])
def test_degenerate_right_hand_sides(b):
    """b = 0 stops before an iteration, NaN at the first check, as before."""
    level, side = 6, 65
    for stored in (False, True):
        mg = H.Multigrid(H.F32, 1, level)
        mg.configure(H.mg_config(tolerance=1e-9, max_outer=20))
        mg.build_q1(0.7)
        if stored:
            mg.set_outer(_operator(side, None))
        rhs = np.zeros(side * side)
        if b == "nan":
            rhs[side * side // 2] = np.nan
        dx = H.DeviceArray(side * side, np.float64)
        dx.zero()
        iters, rd = mg.solve_pcg(H.DeviceArray.from_host(rhs), dx, check=False)
        assert iters == 0 and rd == 0.0, (stored, iters, rd)


def test_rebuilt_with_other_coefficients():
    """A handle built again, with other coefficients or none in between, solves
    as a fresh one."""
    level, side = 7, 129
    b = H.DeviceArray.from_host(uniform_pm1(5, side * side))
    kappas = [H.DeviceArray.from_host(lognormal_cells(s, (side - 1) ** 2), np.float64) for s in (11, 12)]

    def solve(builds):
        mg = H.Multigrid(H.F32, 1, level)
        mg.configure(H.mg_config(tolerance=1e-9, max_outer=60))
        for k in builds:
            if k is None:
                mg.build_q1(0.7)
            else:
                mg.build_q1_coeff(kappas[k], 0.8, 1)
            x = H.DeviceArray(side * side, np.float64)
            x.zero()
            r = mg.solve_pcg(b, x, check=False)
        return r, x.get().tobytes()

    for last in (0, 1, None):
        fresh = solve([last])
        for before in ([0], [1], [None], [0, None], [1, 0]):
            assert solve(before + [last]) == fresh, (before, last)
