"""A point's value does not depend on the call that asks for it: the same bits from the per-point kernel,
the slots-in-lanes traversal, the scalar-slot traversal and the call that allocates nothing.  Points on and
next to the surface, whose FP64 near leaves cancel: a leaf value rounded to the next 2^-40 in one of the
kernels shows in about one of 100,000 of them (|omega| below 1e-3)."""
import numpy as np
import pytest

from lagrange_amd import _lib as L
from lagrange_amd import workloads as W
from lagrange_amd.winding import FastWindingNumber, MultiFastWindingNumber

pytestmark = pytest.mark.gpu

MESHES = {"icosphere 3": lambda: W.icosphere(3), "displaced sphere 6": lambda: W.displaced_sphere(6, 5),
          "icosphere 1": lambda: W.icosphere(1), "open sphere 20": lambda: W.displaced_sphere(20, 3, delete_fraction=0.05)}


def _points(V, F, n, seed):
    rng = np.random.default_rng(seed)
    tri = V[F[rng.integers(0, F.shape[0], n)]].astype(np.float64)
    p = (tri * rng.dirichlet((1, 1, 1), n)[:, :, None]).sum(1)
    d = 10.0 ** rng.uniform(-8, -1, (n, 1)) * rng.standard_normal((n, 3))
    d[: n // 8] = 0.0
    return (p + d).astype(np.float32)


def _noalloc(e, q):
    import torch
    om = torch.empty(q.shape[0], dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    L.check(L.load().fwn_solid_angle_noalloc(e._h(), q.data_ptr(), q.shape[0], om.data_ptr(), None))
    return om


# 250,000: above the slots-in-lanes range of the small meshes; 30,000: within it; 16,384 and 2,048 (from
# host arrays): the per-point kernel
@pytest.mark.parametrize("rel", [1e-4, 0.05])
@pytest.mark.parametrize("name", MESHES)
def test_any_call(name, rel):
    import torch
    V, F = MESHES[name]().f32()
    e = FastWindingNumber((V, F), near_fp64_rel=rel)
    n = 250000
    h = _points(V, F, n, 11)
    q = torch.from_numpy(h).cuda()
    want = e.solid_angle_batch(q).cpu().numpy()
    got = {k: torch.cat([e.solid_angle_batch(x) for x in q.split(k)]).cpu().numpy() for k in (30000, 16384)}
    got["host"] = np.concatenate([e.solid_angle_batch(h[k:k + 2048]) for k in range(0, n, 2048)])
    got["noalloc"] = torch.cat([_noalloc(e, x) for x in q.split(16384)]).cpu().numpy()
    for k, om in got.items():
        np.testing.assert_array_equal(om.view(np.uint32), want.view(np.uint32), err_msg=str(k))


def test_several_meshes():
    meshes = [m().f32() for m in MESHES.values()]
    q = [_points(V, F, 250000 + 17 * k, k) for k, (V, F) in enumerate(meshes)]
    off = np.concatenate([[0], np.cumsum([p.shape[0] for p in q])]).astype(np.int64)
    om = MultiFastWindingNumber(meshes, near_fp64_rel=0.05).solid_angle_batch(points=np.concatenate(q), q_off=off)
    for k, m in enumerate(meshes):
        e = FastWindingNumber(m, near_fp64_rel=0.05)
        each = np.concatenate([e.solid_angle_batch(q[k][a:a + 8192]) for a in range(0, q[k].shape[0], 8192)])
        np.testing.assert_array_equal(om[off[k]:off[k + 1]].view(np.uint32), each.view(np.uint32))
