"""The coarse levels of a V-cycle in one launch against the level-by-level
launches, in a batch pool: the same bits for every parity of the sweep counts
and for slots that enter the launch at each of its levels.
"""
import numpy as np
import pytest

import honei_amd as H
from tests.patterns import lognormal_cells, poisson_system_seeds, uniform_pm1

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


@pytest.mark.parametrize("inner", [H.F32, H.BF16, H.F64])
@pytest.mark.parametrize("n_pre,n_post", [(2, 0), (2, 1), (3, 2), (3, 3), (4, 1)])
def test_coarse_launch_sweeps(n_pre, n_post, inner):
    """Every parity of the sweep counts; slots whose finest level is each of
    the launch's levels and one above it, more slots than one per level."""
    levels, counts = [7, 6, 5, 4, 3, 2], [1, 2, 1, 2, 1, 2]
    got = []
    for fused in (0, 4):
        B = H.Batch(levels, counts, H.batch_config(autotune=0, inner_vtype=inner, n_pre=n_pre, n_post=n_post,
                                                   fused_levels=fused, iters_per_launch=4, max_outer=40))
        keep, slots = [], []
        for c, lv in enumerate(levels):
            for j in range(counts[c]):
                cs, bs = poisson_system_seeds(900 + c, j)
                side = 2 ** lv + 1
                keep.append((H.DeviceArray.from_host(lognormal_cells(cs, (side - 1) ** 2), np.float64),
                             H.DeviceArray.from_host(uniform_pm1(bs, side * side))))
                slots.append(B.slot(c, j))
        B.load_many(slots, [k for k, _ in keep], [b for _, b in keep])
        B.run()
        info = B.poll()
        xs = []
        for g, (_, b) in zip(slots, keep):
            x = H.DeviceArray(b.n, np.float64)
            B.result(g, x)
            xs.append(((info[g].iters, info[g].status, info[g].rel), x.get()))
        got.append(xs)
    for (ia, xa), (ib, xb) in zip(*got):
        assert ia == ib
        assert np.array_equal(xa, xb)
