"""Few-point calls (one wave per point, no sort) against the sorted traversal, which any other launch
shape takes: bit-identical results from host and device arrays at the edges of the path's ranges."""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


def points_of(mesh, n, seed):
    lo, hi = mesh.bbox()
    q = W.uniform_queries(lo, hi, n, seed, scale=1.3)
    q[1::2] = W.near_surface_queries(mesh, n, seed)[1::2]
    return q


# 16: in the kernel arguments; 128: written straight to host memory; 2,049: timed; 16,384: largest
@pytest.mark.parametrize("n", [1, 16, 17, 128, 129, 2049, 16384])
@pytest.mark.parametrize("leaf,width", [(1, 4), (8, 4), (1, 2), (2, 8)])
def test_equals_sorted_traversal(n, leaf, width):
    import torch
    mesh = W.displaced_sphere(48, 5, delete_fraction=0.05)
    e = FastWindingNumber(mesh, leaf_max=leaf, tree_width=width)
    q = points_of(mesh, max(n, 2), 3)[:n]
    oh, ih = e.solid_angle_batch(q, with_inside=True)
    od, id_ = e.solid_angle_batch(torch.from_numpy(q).cuda(), with_inside=True)
    e.set_launch(1, L.FWN_LAUNCH_PERSISTENT)
    big = np.concatenate([q, points_of(mesh, 16400, 9)])  # past the path's range
    ob, ib = e.solid_angle_batch(big, with_inside=True)
    assert np.array_equal(oh.view(np.uint32), ob[:n].view(np.uint32))
    assert np.array_equal(od.cpu().numpy().view(np.uint32), ob[:n].view(np.uint32))
    assert np.array_equal(ih, ib[:n]) and np.array_equal(id_.cpu().numpy(), ib[:n])


def test_walks_past_the_lds_records():
    # beta so large that almost every slot of 5,000 facets is near: records overflow, the wave walks
    # the point again depth first
    mesh = W.displaced_sphere(16, 4)
    e = FastWindingNumber(mesh, accuracy_scale=60.0)
    q = points_of(mesh, 3000, 6)
    few = e.solid_angle_batch(q[:40])
    many = e.solid_angle_batch(q)
    e.set_launch(1, L.FWN_LAUNCH_PERSISTENT)
    ref = e.solid_angle_batch(q)
    assert np.array_equal(few.view(np.uint32), ref[:40].view(np.uint32))
    assert np.array_equal(many.view(np.uint32), ref.view(np.uint32))
