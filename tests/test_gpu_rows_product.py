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


def test_columns_beyond_a_buffer():
    """Columns on both sides of 2^29 and 2^30 (x of 4 GiB and more): byte
    offsets of more than 31 and 32 bits."""
    n, width = MIN_ROWS + 70, 18
    starts = [0, 2 ** 29 - 2048, 2 ** 30 - 2048, 2 ** 30 + 4096]
    cols = starts[-1] + 4096
    stride = 32 * ((n + 31) // 32)
    r = np.arange(n)
    first = np.array(starts)[r // 256 % 4] + r % 3000
    col = first + np.arange(width)[:, None]
    rng = np.random.default_rng(1)
    length = rng.integers(width - 3, width + 1, n)
    used = np.arange(width)[:, None] < length
    Aj, Ax = np.zeros((width, stride), np.uint64), np.zeros((width, stride), np.float32)
    Aj[:, :n] = np.where(used, col, 0)
    Ax[:, :n] = np.where(used, rng.standard_normal((width, n)), 0).astype(np.float32)
    dx, dy = H.DeviceArray(cols, np.float32), H.DeviceArray(n, np.float32)
    dx.zero()
    want = np.zeros(n, np.float32)
    pieces = [rng.standard_normal(4096).astype(np.float32) for _ in starts]
    for c0, p in zip(starts, pieces):
        H.call("honei_hip_upload", H._p(dx.ptr + 4 * c0), p.ctypes.data_as(H._p), p.nbytes, None)
    xv = np.array(pieces)[r // 256 % 4, (r % 3000) + np.arange(width)[:, None]]
    for k in range(width):
        want = np.where(k < length, want + Ax[k, :n] * xv[k], want)
    D = H.DeviceEll(n, cols, stride, width, 1, Aj.reshape(-1), Ax.reshape(-1), length.astype(np.uint64), H.F32)
    D.product(dy, dx)
    assert np.array_equal(dy.get(), want)


@pytest.mark.parametrize("entries", [8, 9])
@pytest.mark.parametrize("scattered", [3, 4, 8])
def test_mixed_work_groups(scattered, entries):
    """Work-groups in which some of the eight wavefronts are scattered, with
    rows on either side of the length from which x is copied; lengths differ
    within a wavefront (0 .. 2 entries, as many of as many more)."""
    n, width = MIN_ROWS + 300, 20
    rng = np.random.default_rng(scattered * 10 + entries)
    stride = 32 * ((n + 31) // 32)
    r = np.arange(n)
    length = np.where(r % 2 == 0, entries, np.where(r % 4 == 1, rng.integers(0, 3, n), 2 * entries))
    wave = r // 64 % 8 < scattered
    col = np.where(wave, rng.integers(0, 6000, (width, n)), r % 3000 + np.arange(width)[:, None])
    used = np.arange(width)[:, None] < length
    Aj, Ax = np.zeros((width, stride), np.uint64), np.zeros((width, stride), np.float32)
    Aj[:, :n] = np.where(used, col, 6000)
    Ax[:, :n] = np.where(used, rng.standard_normal((width, n)), 0).astype(np.float32)
    A = oracle.Ell(n, 6001, stride, width, 1, Aj.reshape(-1), Ax.reshape(-1), length.astype(np.uint64))
    x = rng.standard_normal(6001).astype(np.float32)
    x[6000] = np.nan   # padding only
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray(n, np.float32)
    H.DeviceEll.from_oracle(A).product(dy, dx)
    assert np.array_equal(dy.get(), oracle.product(A, x))
