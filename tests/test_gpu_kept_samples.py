"""Compaction of the kept samples at its edges: sample counts around a wave, a round (256), a tile (4,096)
and the line above which the tiles' counts are scanned first (4,096 tiles).  The kept points equal, in
order, the host-regenerated samples that the engine's own is_inside keeps.
"""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 257, 4095, 4096, 4097, 12288, 100001, 4096 * 4096, 4096 * 4096 + 4097])
def test_kept_samples(n):
    e = FastWindingNumber(W.icosphere(2).f32())
    lo, hi = np.full(3, -1.2, np.float32), np.full(3, 1.2, np.float32)
    u = np.stack([W.rng_uniform(7, 40 + d, n) for d in range(3)], axis=1).astype(np.float32)
    cand = (hi - lo) * u + lo
    want = cand[e.is_inside_batch(cand)]
    np.testing.assert_array_equal(e.sample_inside(n, 7, lo=lo, hi=hi), want)
