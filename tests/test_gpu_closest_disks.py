"""Closest point where the walk's float bounds and slot disks can go wrong, against the brute-force
oracle in double (every facet, Eberly's method).  Both do the same per-triangle arithmetic, and the
walk leaves out only what is farther than its best, so squared distances agree up to what rounding
can make of a triangle left out: 1e-12 relative, and 5e-15 of the largest squared edge (about a
dozen roundings of terms up to 4 L^2); for slivers, whose parameters are off by up to ten roundings
over the squared sine (1e-15 / 1e-6), 1e-7 relative.  A facet differs only where two are equally near.

Points on the surface, deep inside (every slot about as near as the best), at the vertices (exact
ties) and far away; coordinates from 1e-12 to 1e16 and far off the origin; slivers, zero-area and
repeated triangles; tree widths, leaf buckets and both builders; one triangle up to more than the
1,024 of the largest bounded slot.
"""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber

pytestmark = pytest.mark.gpu


def _mesh(kind):
    rng = np.random.default_rng(17)
    V, F = W.displaced_sphere(12, 3, delete_fraction=0.05).f32()
    if kind == "one":
        F = F[:1]
    elif kind == "slivers":  # triangles of sines from about 1e-1 to 1e-3, some of zero area
        P = V[F].astype(np.float64)
        e = P[:, 1] - P[:, 0]
        P[:, 2] = P[:, 0] + 0.5 * e + 10.0 ** -rng.uniform(1, 3, (P.shape[0], 1)) * np.cross(e, P[:, 0])
        P[::11, 2] = P[::11, 0]
        V, F = P.reshape(-1, 3).astype(np.float32), np.arange(3 * P.shape[0], dtype=np.int32).reshape(-1, 3)
    elif kind == "repeated":
        F = np.concatenate([F, F[:300], F[:300]])
    elif kind == "flat":  # coplanar: zero box extents and disks of no thickness
        V = V * np.array([1, 1, 0], np.float32)
    elif kind == "folded":  # two sheets back to back: the slots' normals cancel
        F = np.concatenate([F, F[:, ::-1]])
    return V, np.ascontiguousarray(F, dtype=np.int32)


def _points(V, F, rng):
    tri = V[F[rng.integers(0, F.shape[0], 400)]].astype(np.float64)
    b = rng.dirichlet((1, 1, 1), 400)[:, :, None]
    on = (tri * b).sum(1)
    lo, hi = V.min(0).astype(np.float64), V.max(0).astype(np.float64)
    ext = np.maximum(hi - lo, 1e-30)
    mid = 0.5 * (lo + hi)
    Q = [on, on * (1 + 1e-3), mid + 0.05 * ext * rng.uniform(-1, 1, (300, 3)), V[rng.integers(0, V.shape[0], 200)],
         mid + 2 * ext * rng.uniform(-1, 1, (300, 3)), mid + 1e3 * ext * rng.uniform(-1, 1, (50, 3))]
    return np.concatenate(Q).astype(np.float32)


def _compare(V, F, Q, oracle, rtol=1e-12, **opt):
    d2, fi, cp = FastWindingNumber((V, F), **opt).closest_point(Q)
    od2, ofi, _ = oracle.closest(V, F, Q)
    Vd = V.astype(np.float64)
    edge2 = max(((Vd[F[:, k]] - Vd[F[:, k - 1]]) ** 2).sum(1).max() for k in range(3))
    atol = 5e-15 * edge2
    np.testing.assert_allclose(d2, od2, rtol=rtol, atol=atol)
    for i in np.where(fi != ofi)[0]:
        d, _ = oracle.tri_closest(Vd[F[fi[i], 0]], Vd[F[fi[i], 1]], Vd[F[fi[i], 2]], Q[i])
        assert d == pytest.approx(od2[i], rel=rtol, abs=atol), i


@pytest.mark.parametrize("builder", [L.FWN_TREE_SAH, L.FWN_TREE_LBVH])
@pytest.mark.parametrize("width,leaf", [(2, 1), (4, 1), (4, 8), (8, 3)])
@pytest.mark.parametrize("kind", ["open", "one", "slivers", "repeated", "flat", "folded"])
def test_closest_meshes_and_trees(oracle, kind, width, leaf, builder):
    V, F = _mesh(kind)
    _compare(V, F, _points(V, F, np.random.default_rng(5)), oracle, 1e-7 if kind == "slivers" else 1e-12,
             tree_width=width, leaf_max=leaf, tree_builder=builder)


@pytest.mark.parametrize("scale,offset", [(1e-12, 0.0), (1e-6, 0.0), (1e8, 0.0), (1e16, 0.0), (1.0, 1000.0)])
def test_closest_scales(oracle, scale, offset):
    V, F = _mesh("open")
    V = (V.astype(np.float64) * scale + offset).astype(np.float32)
    _compare(V, F, _points(V, F, np.random.default_rng(6)), oracle)


def test_closest_of_many_waves():
    """Above 2,048 waves the blocks are dealt to the XCDs in runs: with runs and a remainder, the
    distances are those of calls too small for runs."""
    V, F = _mesh("open")
    Q = np.random.default_rng(9).uniform(-1.3, 1.3, (2 * 131072 + 64 * 300 + 5, 3)).astype(np.float32)
    e = FastWindingNumber((V, F))
    want = np.concatenate([e.closest_point(Q[k:k + 50000])[0] for k in range(0, Q.shape[0], 50000)])
    np.testing.assert_array_equal(e.closest_point(Q)[0], want)
