"""The tree build at the edges of its stages: segments of 16 / 17 triangles (row or wave), of 1,024 /
1,025 (one workgroup or level by level), uneven splits that need more levels than a balanced tree,
and many meshes.  Oracle: the CPU restatement's tree, slot by slot."""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu


def soup(n, seed, scale=None):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 1, 3))
    if scale is not None:
        c = c * scale(rng, n)
    V = (c + 0.05 * rng.normal(size=(n, 3, 3))).astype(np.float32).reshape(-1, 3)
    return V, np.arange(3 * n, dtype=np.int32).reshape(-1, 3)


def same_as_restatement(oracle, V, F):
    """Triangle order bit-exact, and the nodes slot by slot (floats within 2e-5 of the slot's largest)."""
    e = FastWindingNumber((V, F))
    slots, tris, roots, _ = e.export_tree()
    R = oracle.Restated(V, F)
    assert 1 + 3 * R.depth < 192  # the engine keeps the SAH tree
    assert np.array_equal(tris.reshape(-1, 12)[:, 9], R.tris.reshape(-1, 12)[:, 9])
    from oracle import oracle as O
    nodes = O.compare_slot_trees(slots, int(roots[0, 0]), int(roots[0, 1]), R.slots, R.root_ns, 4)
    assert nodes == e.tree_info()["num_nodes"] == R.num_nodes


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 18, 33, 1023, 1024, 1025, 2048, 2049, 5000, 70001])
def test_order_equals_restatement(oracle, n):
    V, F = soup(n, n)
    same_as_restatement(oracle, V, F)


@pytest.mark.parametrize("kind", ["geometric", "same", "grid", "two"])
def test_uneven_and_equal_centroids(oracle, kind):
    if kind == "geometric":  # each split peels off a few triangles
        V, F = soup(6000, 1, lambda r, n: np.float64(1.4) ** r.uniform(-60, 20, (n, 1, 1)))
    elif kind == "same":  # middle splits all the way
        V = np.tile(np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32), (3000, 1))
        F = np.arange(9000, dtype=np.int32).reshape(-1, 3)
    elif kind == "grid":  # many equal costs
        rng = np.random.default_rng(5)
        V = rng.integers(0, 12, (9000, 3)).astype(np.float32)
        F = np.arange(9000, dtype=np.int32).reshape(-1, 3)
    else:  # two clusters far apart
        V, F = soup(4000, 2, lambda r, n: np.where(r.random((n, 1, 1)) < 0.001, 1e6, 1.0))
    same_as_restatement(oracle, V, F)


@pytest.mark.parametrize("builder", [L.FWN_TREE_SAH, L.FWN_TREE_LBVH])
def test_many_meshes_equal_single_engines(builder):
    # more meshes than the collapse's first workgroup takes, some without facets
    none = (np.zeros((0, 3), np.float32), np.zeros((0, 3), np.int32))
    meshes = [none if k % 97 == 5 else soup(1 + k % 40, k) for k in range(1100)] + [soup(3000, 7)]
    e = MultiFastWindingNumber(meshes, tree_builder=builder)
    slots, tris, roots, _ = e.export_tree()
    assert np.array_equal(roots[:, 0] < 0, [m[1].shape[0] == 0 for m in meshes])
    rng = np.random.default_rng(3)
    pick = [0, 39, 500, 1099, 1100]
    qs = [rng.uniform(-1.2, 1.2, (20 if k in pick else 0, 3)).astype(np.float32) for k in range(len(meshes))]
    om = e.solid_angle_batch(qs)
    at = 0
    for k in pick:
        one = FastWindingNumber(meshes[k], tree_builder=builder)
        assert np.array_equal(om[at:at + 20], one.solid_angle_batch(qs[k]))
        at += 20


def test_moment_passes_agree():
    V, F = soup(20000, 9)
    a = FastWindingNumber((V, F), moment_pass=L.FWN_MOMENTS_LEVELS).export_tree()
    b = FastWindingNumber((V, F), moment_pass=L.FWN_MOMENTS_CLIMB).export_tree()
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


def test_bad_input_is_still_refused():
    V, F = soup(3000, 4)
    bad = F.copy()
    bad[1234, 1] = V.shape[0]
    with pytest.raises(L.FWNError):
        FastWindingNumber((V, bad))
    W = V.copy()
    W[77, 2] = np.inf
    with pytest.raises(L.FWNError):
        FastWindingNumber((W, F))
