"""The sliced product in steps of eight slots: slices without entries, of one
step, and on either side of a whole number of steps, in windows that end
inside a wavefront's turn of slices; against the CPU product bit for bit.
"""
import numpy as np
import pytest

import honei_amd as H
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    H.init(0)
    yield


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [65, 8 * 64, 8 * 64 + 1, 2048 + 17 * 64 + 5, 2 * 2048])
def test_product(n, dtype):
    rng = np.random.default_rng(n)
    width = 33
    # whole slices of one length (rows are sorted by it within a window)
    length = np.repeat(rng.choice([0, 1, 7, 8, 9, 15, 16, 17, 24, 33], (n + 63) // 64), 64)[:n]
    stride = 32 * ((n + 31) // 32)
    used = np.arange(width)[:, None] < length
    Aj, Ax = np.zeros((width, stride), np.uint64), np.zeros((width, stride), dtype)
    Aj[:, :n] = np.where(used, rng.integers(0, n, (width, n)), 0)
    Ax[:, :n] = np.where(used, rng.standard_normal((width, n)), 0)
    A = oracle.Ell(n, n, stride, width, 1, Aj.reshape(-1), Ax.reshape(-1), length.astype(np.uint64))
    x = rng.standard_normal(n).astype(dtype)
    S = H.Sell(H.DeviceEll.from_oracle(A))
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray(n, dtype)
    S.product(dy, dx)
    assert np.array_equal(dy.get(), oracle.product(A, x))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("window", [1, 2, 1023, 1025, 2048, 2049, 4096, 4097, 10240, 10241, 12288, 12289, 24576, 24577])
def test_windows(window, dtype):
    """Copies of x of one entry to the widest that fits (96 KiB) and one more,
    on either side of each step of the copy; row lengths on either side of the
    steps of four."""
    n, cols, width = 130, 40000, 9
    rng = np.random.default_rng(window)
    length = rng.integers(0, width + 1, n)
    length[0] = width
    stride = 32 * ((n + 31) // 32)
    used = np.arange(width)[:, None] < length
    col = 333 + rng.integers(0, window, (width, n))
    col[0, 0], col[width - 1, 0] = 333, 333 + window - 1
    Aj, Ax = np.zeros((width, stride), np.uint64), np.zeros((width, stride), dtype)
    Aj[:, :n] = np.where(used, col, 0)
    Ax[:, :n] = np.where(used, rng.standard_normal((width, n)), 0)
    A = oracle.Ell(n, cols, stride, width, 1, Aj.reshape(-1), Ax.reshape(-1), length.astype(np.uint64))
    x = rng.standard_normal(cols).astype(dtype)
    x[:333] = x[333 + window:] = np.nan   # never used
    S = H.Sell(H.DeviceEll.from_oracle(A))
    dx, dy = H.DeviceArray.from_host(x), H.DeviceArray(n, dtype)
    S.product(dy, dx)
    assert np.array_equal(dy.get(), oracle.product(A, x))
