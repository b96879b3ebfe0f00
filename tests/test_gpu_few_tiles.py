"""The two-pass sort of calls of few tiles (4,096 points each, at most 128): every point answered once and
in its place.  Results do not depend on the order of the points, so a call equals, bit for bit, calls of
the same points that sort nothing (one wave per point) and calls that sort in three passes.

Counts at the edges of a wave, a tile and the path; points that share one cell, that fall in a few, in
all, and in descending order; several meshes, up to more than the 256 whose number fits the sorted bits.
"""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu


def _points(kind, n, rng):
    q = rng.uniform(-1.3, 1.3, (n, 3))
    if kind == "same":
        q[:] = (0.31, -0.2, 0.7)
    elif kind == "clusters":
        q = 0.02 * q + rng.uniform(-1, 1, (5, 3))[rng.integers(0, 5, n)]
    elif kind == "descending":
        q = q[np.lexsort((q[:, 2], q[:, 1], q[:, 0]))[::-1]]
    return q.astype(np.float32)


@pytest.fixture(scope="module")
def engine():
    return FastWindingNumber(W.displaced_sphere(40, 3, delete_fraction=0.05).f32())


@pytest.mark.parametrize("kind", ["uniform", "same", "clusters", "descending"])
@pytest.mark.parametrize("n", [16385, 20480, 20481, 20543, 131072 + 5])
def test_equals_unsorted_calls(engine, n, kind):
    q = _points(kind, n, np.random.default_rng(n))
    want = np.concatenate([engine.solid_angle_batch(q[k:k + 16384]) for k in range(0, n, 16384)])
    om, inside = engine.solid_angle_batch(q, with_inside=True)
    np.testing.assert_array_equal(om, want)
    np.testing.assert_array_equal(inside.astype(bool), want.astype(np.float64) / (4 * np.pi) > 0.5)


@pytest.mark.parametrize("n", [128 * 4096 - 1, 128 * 4096, 128 * 4096 + 1])
def test_both_sides_of_the_line(engine, n):
    q = _points("uniform", 128 * 4096 + 4096, np.random.default_rng(1))  # the whole sorts in three passes
    np.testing.assert_array_equal(engine.solid_angle_batch(q[:n]), engine.solid_angle_batch(q)[:n])


@pytest.mark.parametrize("meshes", [2, 3, 255, 256, 257, 400])
def test_several_meshes(meshes):
    rng = np.random.default_rng(meshes)
    kinds = [W.icosphere(2).f32(), W.icosphere(4).f32(), W.displaced_sphere(5, 2).f32()]
    m = [kinds[k % 3] for k in range(meshes)]
    cnt = rng.integers(0, 2 * 40000 // meshes, meshes)
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    q = _points("uniform", int(off[-1]), rng)
    om = MultiFastWindingNumber(m).solid_angle_batch(points=q, q_off=off)
    single = [FastWindingNumber(k) for k in kinds]
    for k in range(meshes):
        if cnt[k]:
            np.testing.assert_array_equal(om[off[k]:off[k + 1]], single[k % 3].solid_angle_batch(q[off[k]:off[k + 1]]))
