"""y = A x of wide float rows, one lane per row: rows in registers with x from
LDS, from global memory, or in steps, against the CPU product bit for bit.
"""
import numpy as np
import pytest

import honei_amd as H
import oracle

pytestmark = pytest.mark.gpu

MIN_ROWS = 98304   # smallest product that takes the wide-row kernel
WINDOW = 9216      # widest column window that is copied


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


def _matrix(n, cols, width, pattern):
    """Rows of 0 .. width entries: columns within the row's own 512-row block
    and `pattern` beyond it (window 512 + pattern), anywhere, or consecutive;
    padding holds the column of a NaN in x that no row uses."""
    rng = np.random.default_rng(n * 31 + width)
    stride = 32 * ((n + 31) // 32)
    length = rng.integers(0, width + 1, n)
    length[:2000] = 0                      # work-groups without an entry
    length[-1] = width
    r = np.arange(n)
    if pattern == "everywhere":
        cols_ = rng.integers(0, cols - 1, (width, n))
    elif pattern == "band":
        cols_ = np.clip(r + np.arange(width)[:, None] - width // 2, 0, cols - 2)
    else:
        base = np.minimum(r // 512 * 512, cols - 1 - pattern)
        cols_ = base + rng.integers(0, pattern, (width, n))
        cols_[0], cols_[1] = base, base + pattern - 1   # the whole window is used
    used = np.arange(width)[:, None] < length
    Aj = np.full((width, stride), cols - 1, np.uint64)
    Ax = np.zeros((width, stride), np.float32)
    Aj[:, :n] = np.where(used, cols_, cols - 1)
    Ax[:, :n] = np.where(used, rng.standard_normal((width, n)), 0).astype(np.float32)
    A = oracle.Ell(n, cols, stride, width, 1, Aj.reshape(-1), Ax.reshape(-1), length.astype(np.uint64))
    x = rng.standard_normal(cols).astype(np.float32)
    x[cols - 1] = np.nan
    x[cols // 2] = np.inf
    return A, x


CASES = [(width, n, p) for width, n in [(17, MIN_ROWS), (24, MIN_ROWS + 1), (25, MIN_ROWS + 511), (28, MIN_ROWS + 513)]
         for p in [WINDOW, WINDOW + 1, 700, "everywhere", "band"]]


@pytest.mark.parametrize("width,n,pattern", CASES + [(17, MIN_ROWS - 1, 700), (16, MIN_ROWS, 700), (29, MIN_ROWS, 700)])
def test_product(width, n, pattern):
    A, x = _matrix(n, n + 3, width, pattern)
    want = oracle.product(A, x)
    D = H.DeviceEll.from_oracle(A)
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray(n, np.float32)
    D.product(dy, dx)
    assert np.array_equal(dy.get(), want, equal_nan=True)
    # a range of rows, written from its first row on
    first, last = 77, n - 130
    if last - first >= MIN_ROWS - 512:
        part = H.DeviceArray(last - first, np.float32)
        D.product(part, dx, row_start=first, row_end=last)
        assert np.array_equal(part.get(), want[first:last], equal_nan=True)


@pytest.mark.parametrize("pattern", [700, "everywhere", "band"])
def test_first_two_rows_of_a_wavefront(pattern):
    """Only lanes 0 and 1 have entries: what the work-group decides on is the
    one pair of neighbouring rows a wavefront has."""
    n, width = MIN_ROWS + 64, 27
    A, x = _matrix(n, n + 3, width, pattern)
    length = A.Arl.copy()
    length[np.arange(n) % 64 > 1] = 0
    A = oracle.Ell(n, n + 3, A.stride, width, 1, A.Aj, A.Ax, length)
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray(n, np.float32)
    H.DeviceEll.from_oracle(A).product(dy, dx)
    assert np.array_equal(dy.get(), oracle.product(A, x), equal_nan=True)
