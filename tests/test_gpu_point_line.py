"""Which device calls of one mesh run one wave per point: up to 16,384 points while their walks fit into
the LDS records (a line on accuracy scale and triangles), 8,192 with buckets, 2,048 beyond.  Such a call
reports one kernel, so its traversal takes its whole device time; the sorted traversals' calls take longer
than their traversal.  The values are those of small calls on either side."""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


# spheres of 20 nu^2 triangles, scale^2 log2(F / 64) = 75, 86.8, 92.9 and 133 for the first and last ones
@pytest.mark.parametrize("nu,scale,leaf,line", [
    (32, 3.0, 1, 16384), (64, 2.9, 1, 16384), (64, 3.0, 1, 2048), (32, 4.0, 1, 2048), (8, 3.0, 1, 16384),
    (8, 3.1, 1, 2048), (32, 2.0, 3, 8192), (1, 3.0, 1, 16384), (1, 8.0, 8, 2048)])
def test_line(nu, scale, leaf, line):
    import torch
    mesh = W.displaced_sphere(nu, 5)
    e = FastWindingNumber(mesh, accuracy_scale=scale, leaf_max=leaf)
    lo, hi = mesh.bbox()
    q = W.uniform_queries(lo, hi, 16400, 3, scale=1.2)
    q[1::2] = W.near_surface_queries(mesh, 16400, 3)[1::2]
    d = torch.from_numpy(np.ascontiguousarray(q, np.float32)).cuda()
    want = torch.cat([e.solid_angle_batch(x) for x in d.split(2000)])
    for n in (line, line + 1):
        om = e.solid_angle_batch(d[:n])
        traverse, total = e.last_timing()
        assert (traverse == total) == (n <= line)
        assert torch.equal(om, want[:n])
