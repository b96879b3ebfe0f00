import numpy as np
import pytest

from lagrange_amd.bounds import column_bounds


# below and above two blocks of 128 rows, whole blocks and remainders, a strided view, NaN
@pytest.mark.parametrize("n", [1, 127, 255, 256, 257, 384, 1000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_equals_numpy(n, dtype):
    V = np.random.default_rng(n).normal(size=(n, 6)).astype(dtype)
    for X in (np.ascontiguousarray(V[:, :3]), V[:, 1:4]):
        lo, hi = column_bounds(X)
        assert lo.dtype == dtype and np.array_equal(lo, X.min(axis=0)) and np.array_equal(hi, X.max(axis=0))
    X = np.ascontiguousarray(V[:, :3])
    X[n // 2, 1] = np.nan
    assert np.array_equal(column_bounds(X)[0], X.min(axis=0), equal_nan=True)
