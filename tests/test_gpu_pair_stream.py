"""The paired row passes that march down column strips (large levels) against
one launch per pass, and the CG direction that marches down its tiles against
the tile launch, in a batch pool: the same bits while all systems run and when
the last few do.
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


def _same(levels, counts, **variants):
    """Both values of the one option in `variants` give the same results."""
    (option, values), = ((k, v) for k, v in variants.items() if isinstance(v, tuple))
    rest = {k: v for k, v in variants.items() if k != option}
    got = []
    for value in values:
        B = H.Batch(levels, counts, H.batch_config(autotune=0, iters_per_launch=4, max_outer=40, **rest,
                                                   **{option: value}))
        keep, slots = [], []
        for c, lv in enumerate(levels):
            for j in range(counts[c]):
                if j >= 20:   # the earlier systems again
                    keep.append(keep[-20])
                    slots.append(B.slot(c, j))
                    continue
                cs, bs = poisson_system_seeds(400 + c, j)
                side = 2 ** lv + 1
                # systems that need more iterations than the others: the last to run
                cells = lognormal_cells(cs, (side - 1) ** 2) ** (1.5 if j == 0 else 1.0)
                keep.append((H.DeviceArray.from_host(cells, np.float64),
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
        assert np.isfinite(xa).all() and xa.any()


# launches of many tiles on one level, on each level, and with all levels'
# systems together; one system short of the rule on its finest level; enough
# systems for medium and for long segments (shorter ones as systems finish)
@pytest.mark.parametrize("levels,counts", [([7], [18]), ([7], [17]), ([8], [6]), ([9, 8, 7], [2, 4, 14]),
                                           ([7], [130]), ([7], [230])])
@pytest.mark.parametrize("inner", [H.F32, H.BF16, H.F64])
def test_pairs(inner, levels, counts):
    _same(levels, counts, inner_vtype=inner, pair_sweeps=(0, 1))


# 1024 tiles (15, 45 and 162 a system of levels 7, 8 and 9) and fewer, every
# band of rows short of its full height among them
@pytest.mark.parametrize("levels,counts", [([7], [69]), ([7], [68]), ([9, 8, 7], [4, 6, 8]), ([8, 5, 3], [20, 80, 60])])
@pytest.mark.parametrize("inner", [H.F32, H.F64])
def test_direction(inner, levels, counts):
    _same(levels, counts, inner_vtype=inner, matrix_free=(0, 1))
