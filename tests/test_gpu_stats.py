"""Work counters: every point of the call is answered, whatever launch shape the engine has."""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves,mode", [(1, L.FWN_LAUNCH_GRID), (2, L.FWN_LAUNCH_GRID), (8, L.FWN_LAUNCH_GRID),
                                        (4, L.FWN_LAUNCH_PERSISTENT)])
def test_stats_answer_every_point(waves, mode):
    mesh = W.displaced_sphere(16, 2)
    lo, hi = mesh.bbox()
    q = W.uniform_queries(lo, hi, 5003, 7, scale=1.3)
    e = FastWindingNumber(mesh)
    e.set_launch(waves, mode)
    om, stats = e.query_stats(q)  # the engine's first call: nothing of an earlier one lies in its outputs
    assert (stats[:, 0] > 0).all()
    want, counts = FastWindingNumber(mesh).query_stats(q)
    np.testing.assert_array_equal(om, want)
    np.testing.assert_array_equal(stats, counts)
