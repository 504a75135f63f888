"""Multigrid cycles from a zero start (initial_zero) and more than one cycle a
call, against the CPU path: every cycle after the first smooths the defect of
the iterate, not the right-hand side it started from.
"""
import numpy as np
import pytest

import honei_amd as H
import oracle
from tests.patterns import uniform_pm1

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _problem(side):
    A = oracle.q1_matrix(side)
    xt = uniform_pm1(3, side * side)
    return A, xt, oracle.product(A, xt)


# levels in the coarse launch and above it (FP32 and bf16 from 7, FP64 from 6);
# stored: the same solve on the stored matrices, no structure assumed
@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("level,n_max_iter", [(4, 2), (6, 3), (8, 2), (8, 4)])
def test_mixed(level, n_max_iter, stored):
    side = 2 ** level + 1
    A, xt, b = _problem(side)
    kw = dict(n_max_iter=n_max_iter, tolerance=1e-8, initial_zero=True, zero_inner_start=True)
    xo, outer_o, inner_o, _ = oracle.mg_mixed(oracle.q1_hierarchy(level, dtype=np.float32),
                                              oracle.mg_config(1, level, **kw), A, b)
    mg = H.Multigrid(H.F32, 1, level)
    mg.configure(H.mg_config(max_outer=60, **kw))
    mg.build_q1(0.7)
    if stored:
        mg.set_outer(A)
    db, dx = H.DeviceArray.from_host(b), H.DeviceArray(side * side, np.float64)
    dx.zero()
    outer, inner, rd = mg.solve_mixed(db, dx, check=False)
    assert (outer, inner) == (outer_o, inner_o)
    assert rd < 1e-8
    # both within 1e-8 (relative defect) of the same solution, as the other
    # mixed solves are compared
    assert np.abs(dx.get() - xo).max() <= 1e-6 * np.abs(xo).max()
    assert np.abs(dx.get() - xt).max() < 1e-6


@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("level", [4, 6, 8])
def test_fixed(level, stored):
    side = 2 ** level + 1
    A, xt, b = _problem(side)
    kw = dict(n_max_iter=50, tolerance=1e-10, initial_zero=True)
    xo, it_o, _ = oracle.mg_fixed(oracle.q1_hierarchy(level, dtype=np.float64), oracle.mg_config(1, level, **kw), b)
    mg = H.Multigrid(H.F64, 1, level)
    mg.configure(H.mg_config(**kw))
    mg.build_q1(0.7)
    if stored:
        mg.set_outer(A)
    db, dx = H.DeviceArray.from_host(b), H.DeviceArray(side * side, np.float64)
    dx.zero()
    it, _ = mg.solve_fixed(db, dx)
    assert it == it_o
    assert np.abs(dx.get() - xo).max() <= 1e-9 * max(1.0, np.abs(xo).max())
    assert np.abs(dx.get() - xt).max() < 1e-8
