"""The slots-in-lanes traversal (default launch shape, sparse calls) against the scalar-slot one
(any other launch shape): the same terms in the same order, so bit-identical results."""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu


def both(engine, call):
    engine.set_launch(1, L.FWN_LAUNCH_GRID)
    a = call()
    engine.set_launch(1, L.FWN_LAUNCH_PERSISTENT)
    b = call()
    return a, b


def mixed_points(mesh, n, seed):
    """Uniform points of the box x1.3 and points on and next to the surface, interleaved."""
    lo, hi = mesh.bbox()
    q = W.uniform_queries(lo, hi, n, seed, scale=1.3)
    q[1::2] = W.near_surface_queries(mesh, n, seed)[1::2]
    q[::97] = mesh.vertices[np.arange(0, n, 97) % mesh.num_vertices]
    return q


# 16,385 is the smallest such call of one mesh; 16 k + {0, 1, 15} points end in a full or partial wave
@pytest.mark.parametrize("n", [16385, 16399, 16400, 30001])
@pytest.mark.parametrize("leaf", [1, 3, 8])
@pytest.mark.parametrize("nu,delete", [(1, 0.0), (3, 0.5), (32, 0.0), (64, 0.05)])
def test_equals_scalar_slot_traversal(n, leaf, nu, delete):
    mesh = W.displaced_sphere(nu, 7, delete_fraction=delete)
    e = FastWindingNumber(mesh, leaf_max=leaf)
    q = mixed_points(mesh, n, 11)
    (oa, ia), (ob, ib) = both(e, lambda: e.solid_angle_batch(q, with_inside=True))
    assert np.array_equal(oa.view(np.uint32), ob.view(np.uint32))
    assert np.array_equal(ia, ib)


def test_fp64_queue_wraps():
    # every point has many FP64 leaves (tau of the size of the mesh): the queue fills and drains
    mesh = W.displaced_sphere(12, 3)
    e = FastWindingNumber(mesh, near_fp64_rel=0.3)
    q = mixed_points(mesh, 17000, 5)
    a, b = both(e, lambda: e.solid_angle_batch(q))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_multi_mesh_with_empty_and_single_facet_meshes():
    tri = W.Mesh(np.array([[0.0, 0, 0], [1, 0, 0], [0, 1, 0]]), np.array([[0, 1, 2]]))
    none = W.Mesh(np.zeros((0, 3)), np.zeros((0, 3), np.int64))
    meshes = [W.displaced_sphere(20, 1), none, tri, W.torus(40, 12)]
    e = MultiFastWindingNumber(meshes)
    qs = [mixed_points(meshes[0], 1501, 2), W.uniform_queries(-np.ones(3), np.ones(3), 33, 3),
          W.uniform_queries(-np.ones(3), np.ones(3), 17, 4), mixed_points(meshes[3], 900, 5)]
    (oa, ia), (ob, ib) = both(e, lambda: e.solid_angle_batch(qs, with_inside=True))
    assert np.array_equal(oa.view(np.uint32), ob.view(np.uint32))
    assert np.array_equal(ia, ib)
