"""Host calls of up to 2,048 points: one kernel, whose waves store their results to host memory; larger
ones collect them on the device first.  Equal results either way."""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


def kernels(call):
    """Names of the kernels that the call launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    return [ev.name for ev in p.events() if "fwn" in ev.name]


@pytest.mark.parametrize("n,publishes", [(17, 0), (129, 0), (200, 0), (2048, 0), (2049, 1)])
def test_kernels_of_a_host_call(n, publishes):
    mesh = W.displaced_sphere(16, 2)
    e = FastWindingNumber(mesh)
    lo, hi = mesh.bbox()
    q = W.uniform_queries(lo, hi, n, 7, scale=1.3)
    om, inside = e.solid_angle_batch(q, with_inside=True)
    names = kernels(lambda: e.solid_angle_batch(q, with_inside=True))
    assert sum("k_point_bfs" in k for k in names) == 1
    assert sum("k_publish" in k for k in names) == publishes and len(names) == 1 + publishes
    om_1 = np.concatenate([e.solid_angle_batch(q[k:k + 16]) for k in range(0, n, 16)])
    np.testing.assert_array_equal(om, om_1)
    np.testing.assert_array_equal(inside, om_1.astype(np.float64) / (4 * np.pi) > 0.5)
