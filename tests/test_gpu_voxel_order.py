"""The voxel box's own order of waves (4 x 4 x 4 blocks, cut short at the far faces) in place of a sort:
every voxel answered once and in its place.  Results do not depend on the order, so each box equals
the list of its voxels, which is sorted, bit for bit.  Boxes of one and of several blocks with every
kind of cut face, lines and sheets, and launch shapes whose smallest boxes take the sorted path.
"""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(27, 26, 25), (28, 24, 32), (1, 1, 20001), (20001, 1, 1), (1, 20001, 1), (3, 5, 1201),
                                  (130, 131, 1), (2, 97, 102), (401, 2, 33), (64, 64, 66)], ids=str)
def test_box_equals_list(dims):
    V, F = W.displaced_sphere(8, 3, delete_fraction=0.05).f32()
    e = FastWindingNumber((V, F))
    vs = 2.4 / max(dims)
    lo = [-(d // 2) for d in dims]
    z, y, x = np.meshgrid(*(np.arange(d) for d in dims[::-1]), indexing="ij")
    ijk = np.stack([x.ravel() + lo[0], y.ravel() + lo[1], z.ravel() + lo[2]], 1).astype(np.int32)
    ins, om = e.sign_voxel_box(lo, dims, vs, with_omega=True)
    want, om_want = e.sign_voxels(ijk, vs, with_omega=True)
    np.testing.assert_array_equal(om.ravel(), om_want)
    np.testing.assert_array_equal(ins.ravel(), want)


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 6, 7), (13, 14, 15), (17, 3, 50)], ids=str)
def test_other_launch_shapes(dims):
    V, F = W.icosphere(6).f32()
    e = FastWindingNumber((V, F))
    lo = [-(d // 2) for d in dims]
    ins, om = e.sign_voxel_box(lo, dims, 0.15, with_omega=True)
    e.set_launch(4, 0)
    ins4, om4 = e.sign_voxel_box(lo, dims, 0.15, with_omega=True)
    np.testing.assert_array_equal(om4, om)
    np.testing.assert_array_equal(ins4, ins)
