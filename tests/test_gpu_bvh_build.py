"""The device BVH build at the sizes where its paths change: one wave (up to
64 triangles), one workgroup (up to 4,096), several workgroups per task, the
edges of their chunks, equal and collinear centroids. Every build holds every
triangle once, its boxes contain them, and its closest hits equal the
host-built tree's."""
import numpy as np
import pytest

import reina_rt
from reina_rt import abi
from reina_rt.scene import Material, ModelData, Scene

pytestmark = pytest.mark.gpu


def _arrays(tris):
    n = len(tris)
    v = np.concatenate([tris.reshape(-1, 3), np.ones((3 * n, 1))], 1).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32)
    s = Scene()
    s.add_object(ModelData(v, idx, np.tile(np.eye(3, dtype=np.float32), (3 * n, 1, 1)), idx.copy()), np.eye(4),
                 Material(materialIdx=0))
    return s.build_arrays()


def _soup(n, kind):
    rng = np.random.default_rng(n)
    base = np.array([[0, 0, 0], [0.1, 0, 0], [0, 0.1, 0]], float)
    if kind == "same":
        return np.tile(base, (n, 1, 1))
    if kind == "line":
        return base[None] + np.arange(n)[:, None, None] * np.array([0.3, 0.0, 0.0])
    return rng.random((n, 1, 3)) * 4 + 0.1 * rng.normal(size=(n, 3, 3))


def _check_tree(dev, n):
    nodes, tris = dev.export_bvh()
    nodes = nodes.reshape(-1, 256)
    box = nodes[:, :192].copy().view(np.float32).reshape(-1, 3, 2, 8)          # axis, lo/hi, slot
    child = nodes[:, 192:196].copy().view(np.uint32).reshape(-1)
    trib = nodes[:, 196:200].copy().view(np.uint32).reshape(-1)
    meta = nodes[:, 200:208]
    t = tris.reshape(-1, 3, 4)
    ids = t[:, 0, 3].copy().view(np.uint32)
    assert np.array_equal(np.sort(ids), np.arange(n))
    seen = np.zeros(n, int)
    stack, visited = [0], 0
    while stack:
        k = stack.pop()
        visited += 1
        for s in range(8):
            m = int(meta[k, s])
            if m == 0:
                continue
            if m & 0x80:
                c = int(child[k] & 0xFFFFFF) + (m & 0x7F)
                used = meta[c] != 0
                assert (box[c][:, 0][:, used].min(1) >= box[k, :, 0, s]).all()
                assert (box[c][:, 1][:, used].max(1) <= box[k, :, 1, s]).all()
                stack.append(c)
            else:
                first = int(trib[k] & 0xFFFFFF) + (m & 31)
                p = t[first:first + (m >> 5), :, :3]
                assert (p.min((0, 1)) >= box[k, :, 0, s]).all() and (p.max((0, 1)) <= box[k, :, 1, s]).all()
                seen[first:first + (m >> 5)] += 1
    assert visited == len(nodes) and (seen == 1).all()


@pytest.mark.parametrize("n,kind", [(1, "soup"), (2, "soup"), (64, "soup"), (65, "soup"), (4096, "soup"),
                                    (4097, "soup"), (5120, "soup"), (5121, "soup"), (20011, "soup"), (65, "same"),
                                    (9001, "same"), (63, "line"), (9000, "line")])
def test_device_build_sizes(cuda, n, kind):
    torch = cuda
    arrays = _arrays(_soup(n, kind))
    a, b = reina_rt.DeviceScene(arrays), reina_rt.DeviceScene(arrays, flags=abi.BUILD_HOST)
    _check_tree(a, n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    rays = torch.zeros((4096, 8), device="cuda")
    rays[:, 0:3] = torch.rand((4096, 3), device="cuda", generator=g) * 4 - torch.tensor([0.0, 0.0, 6.0], device="cuda")
    rays[:, 4:7] = torch.nn.functional.normalize(
        torch.randn((4096, 3), device="cuda", generator=g) * 0.3 + torch.tensor([0.0, 0.0, 1.0], device="cuda"), dim=1)
    rays[:, 7] = 1e4
    ha, hb = torch.zeros((4096, 4), device="cuda"), torch.zeros((4096, 4), device="cuda")
    a.intersect(rays.data_ptr(), ha.data_ptr(), 4096)
    b.intersect(rays.data_ptr(), hb.data_ptr(), 4096)
    torch.cuda.synchronize()
    assert torch.equal(ha.view(torch.int32), hb.view(torch.int32))
    a.close()
    b.close()
