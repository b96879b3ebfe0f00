"""The batched traversal's FP64 near leaves (queued in LDS, 64 evaluated at a time) against the
per-point kernel, which sums each point's own leaves.  Both add the same leaves in 2^-40 fixed point
and the same FP32 terms in the same order, so the results of points near the surface, which are not
small, are equal bit for bit.

A large near_fp64_rel makes every near leaf an FP64 leaf: a node can then queue 64 entries for each of
its slots (2, 4 and 8 wide).  Point counts around a wave and a partly filled last one, leaf buckets,
both stack sizes, every launch shape, and points of several meshes.
"""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu


def _points(V, F, n, seed):
    rng = np.random.default_rng(seed)
    tri = V[F[rng.integers(0, F.shape[0], n)]].astype(np.float64)
    p = (tri * rng.dirichlet((1, 1, 1), n)[:, :, None]).sum(1)
    d = 10.0 ** rng.uniform(-8, -1, (n, 1)) * rng.standard_normal((n, 3))
    d[: n // 8] = 0.0
    return (p + d).astype(np.float32)


def _each(e, q):
    return np.concatenate([e.solid_angle_batch(q[k:k + 8192]) for k in range(0, q.shape[0], 8192)])


@pytest.mark.parametrize("rel", [0.0, 1e-3, 10.0])
@pytest.mark.parametrize("opt", [dict(tree_width=2), dict(tree_width=4), dict(tree_width=8), dict(leaf_max=8),
                                 dict(tree_width=8, leaf_max=3, tree_builder=L.FWN_TREE_LBVH)], ids=str)
def test_queue_equals_per_point(opt, rel):
    V, F = W.displaced_sphere(10, 3, delete_fraction=0.05).f32()
    e = FastWindingNumber((V, F), near_fp64_rel=rel, **opt)
    for n in (16385, 16385 + 63, 300001):  # the last above the slots-in-lanes range
        q = _points(V, F, n, n)
        om, inside = e.solid_angle_batch(q, with_inside=True)
        want = _each(e, q)
        np.testing.assert_array_equal(om, want)
        np.testing.assert_array_equal(inside.astype(bool), want.astype(np.float64) / (4 * np.pi) > 0.5)


@pytest.mark.parametrize("waves,mode", [(1, 1), (2, 0), (4, 0), (8, 0), (4, 1), (8, 1)])
def test_queue_in_every_launch_shape(waves, mode):
    V, F = W.icosphere(12).f32()
    e = FastWindingNumber((V, F), near_fp64_rel=0.05)
    q = _points(V, F, 30001, 5)
    want = _each(e, q)
    e.set_launch(waves, mode)
    np.testing.assert_array_equal(e.solid_angle_batch(q), want)


def test_queue_with_several_meshes():
    """Against the same traversal on an engine of each mesh (250,000 points of a small mesh are above
    the slots-in-lanes range).  Not against the per-point kernel: its compilation of the FP64 formula may
    round a leaf's value to the next 2^-40, which shows where a point's terms cancel to 1e-3 and less."""
    meshes = [W.icosphere(3).f32(), W.displaced_sphere(6, 5).f32(), W.icosphere(1).f32()]
    q = [_points(V, F, 250000 + 17 * k, k) for k, (V, F) in enumerate(meshes)]
    off = np.concatenate([[0], np.cumsum([p.shape[0] for p in q])]).astype(np.int64)
    mm = MultiFastWindingNumber(meshes, near_fp64_rel=0.05)
    om = mm.solid_angle_batch(points=np.concatenate(q), q_off=off)
    for k, m in enumerate(meshes):
        np.testing.assert_array_equal(om[off[k]:off[k + 1]],
                                      FastWindingNumber(m, near_fp64_rel=0.05).solid_angle_batch(q[k]))


@pytest.mark.parametrize("n", [499999, 500000, 500001, 640001])
@pytest.mark.parametrize("where", ["box", "layer", "one"])
def test_calls_that_look_at_their_spread(where, n):
    """Above 500,000 points of one mesh the kernel is chosen by how the points spread over the mesh's box:
    the same results on both sides of the line and of the choice (24,000 cbrt(F) = 643,000 here)."""
    V, F = W.icosphere(31).f32()
    e = FastWindingNumber((V, F))
    rng = np.random.default_rng(n)
    q = rng.uniform(-1.1, 1.1, (n, 3))
    if where == "layer":
        q *= 1.05 / np.linalg.norm(q, axis=1, keepdims=True)
    elif where == "one":
        q[:] = (0.4, 0.1, -0.2)
    q = q.astype(np.float32)
    take = rng.integers(0, n, 8192)
    np.testing.assert_array_equal(e.solid_angle_batch(q)[take], e.solid_angle_batch(q[take]))
