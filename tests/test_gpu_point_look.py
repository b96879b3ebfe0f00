"""Which traversal calls above 450,000 points take: slots in lanes for points that spread over the mesh's box
(random, regular grids of powers of two, dense voxel boxes) or, several meshes or few enough points, lie near
the surface; the scalar-slot one for layers off the surface and boxes far smaller than the mesh.  By the
kernels that run; the values are those of small calls."""
import numpy as np
import pytest

from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu


def traversal(call):
    """(result, name of the traversal that ran)"""
    import torch
    from torch.profiler import ProfilerActivity, profile
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        r = call()
        torch.cuda.synchronize()
    names = [ev.name for ev in p.events() if "k_traverse" in ev.name]
    assert len(names) == 1, names
    return r, "quad" if "k_traverse_quad" in names[0] else "scalar"


def layer(V, F, n, off, seed):
    rng = np.random.default_rng(seed)
    T = V[F[rng.integers(0, F.shape[0], n)]].astype(np.float64)
    nn = np.cross(T[:, 1] - T[:, 0], T[:, 2] - T[:, 0])
    nn /= np.linalg.norm(nn, axis=1, keepdims=True)
    return ((T * rng.dirichlet((1, 1, 1), n)[:, :, None]).sum(1) + off * nn).astype(np.float32)


def grid(dims):
    t = [np.linspace(-1.2, 1.2, k) for k in dims]
    z, y, x = np.meshgrid(t[2], t[1], t[0], indexing="ij")
    return np.stack([x, y, z], -1).reshape(-1, 3).astype(np.float32)


# F = 20,480: the line is 657,000 points
POINTS = {"random": (lambda V, F: np.random.default_rng(1).uniform(-1.2, 1.2, (500001, 3)).astype(np.float32), "quad"),
          "64 x 64 x 128": (lambda V, F: grid((64, 64, 128)), "quad"),
          "128 x 128 x 32": (lambda V, F: grid((128, 128, 32)), "quad"),
          "on the surface": (lambda V, F: layer(V, F, 480000, 0.0, 2), "quad"),
          "on the surface, more": (lambda V, F: layer(V, F, 640000, 0.0, 2), "scalar"),
          "layer": (lambda V, F: layer(V, F, 480000, 0.3, 3), "scalar"),
          "layer, few": (lambda V, F: layer(V, F, 449999, 0.3, 3), "quad"),
          "one place": (lambda V, F: np.full((500000, 3), 0.3, np.float32), "scalar"),
          "not a number": (lambda V, F: np.full((450001, 3), np.nan, np.float32), "scalar"),
          "past the line": (lambda V, F: np.random.default_rng(1).uniform(-1.2, 1.2, (700001, 3)).astype(np.float32), "scalar")}


@pytest.mark.parametrize("name", POINTS)
def test_one_mesh(name):
    import torch
    V, F = W.icosphere(32).f32()
    e = FastWindingNumber((V, F))
    points, want = POINTS[name]
    q = points(V, F)
    d = torch.from_numpy(q).cuda()
    om, kernel = traversal(lambda: e.solid_angle_batch(d))
    assert kernel == want
    take = np.random.default_rng(4).integers(0, q.shape[0], 8192)
    np.testing.assert_array_equal(om.cpu().numpy()[take].view(np.uint32),
                                  e.solid_angle_batch(q[take]).view(np.uint32))


@pytest.mark.parametrize("where,want", [("random", "quad"), ("surface", "quad"), ("layer", "scalar")])
@pytest.mark.parametrize("first", [20000, 200000])
def test_several_meshes(where, want, first):
    """The mesh with the most points is looked at (the fourth or the first); one mesh has neither facets nor
    points.  The line is 24,000 cbrt(mean F) + 2 F > 900,000 points."""
    import torch
    meshes = [W.displaced_sphere(40 + 8 * k, k).f32() for k in range(4)]
    meshes.insert(2, (np.zeros((0, 3), np.float32), np.zeros((0, 3), np.int32)))
    n = [first, 100001, 0, 180003, 200001 - first // 2]
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    assert 450000 < off[-1] < 24000 * np.cbrt(sum(F.shape[0] for _, F in meshes) / 5)
    qs = []
    for k, (V, F) in enumerate(meshes):
        if where == "random" or n[k] == 0:
            qs.append(np.random.default_rng(k).uniform(-1.3, 1.3, (n[k], 3)).astype(np.float32))
        else:
            qs.append(layer(V, F, n[k], 0.0 if where == "surface" else 0.5, k))
    e = MultiFastWindingNumber(meshes)
    d = torch.from_numpy(np.concatenate(qs)).cuda()
    om, kernel = traversal(lambda: e.solid_angle_batch(points=d, q_off=off))
    assert kernel == want
    om = om.cpu().numpy()
    for k, m in enumerate(meshes):
        take = np.random.default_rng(4).integers(0, n[k], 4096) if n[k] else np.zeros(0, np.int64)
        got = FastWindingNumber(m).solid_angle_batch(qs[k][take])
        np.testing.assert_array_equal(om[off[k] + take].view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("lo,dims,size,want", [((-40,) * 3, (80, 80, 80), 0.03, "quad"),
                                               ((-40,) * 3, (80, 80, 80), 0.002, "scalar"),
                                               ((-100, -100, 0), (200, 200, 12), 0.012, "scalar"),
                                               ((-300,) * 3, (80, 80, 80), 0.03, "scalar")])
def test_voxel_boxes(lo, dims, size, want):
    mesh = W.icosphere(32)
    e = FastWindingNumber(mesh)
    (inside, om), kernel = traversal(lambda: e.sign_voxel_box(lo, dims, size, with_omega=True, device="cuda"))
    assert kernel == want
    take = np.random.default_rng(1).integers(0, om.numel(), 4000)
    z, y, x = np.unravel_index(take, om.shape)
    v = np.stack([x, y, z], -1) + np.array(lo)
    q = (v * size + size * 0.5).astype(np.float32)
    np.testing.assert_array_equal(om.reshape(-1).cpu().numpy()[take].view(np.uint32), e.solid_angle_batch(q).view(np.uint32))
