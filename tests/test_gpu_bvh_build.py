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


def _flatten(arrays):
    """world = ((c0 x + c1 y) + c2 z) + c3 in float32, instance by instance."""
    out = []
    v, idx = arrays["vertices"].reshape(-1, 4), arrays["indices"]
    for i in arrays["instances"]:
        m = arrays["models"][i["modelID"]]
        c = i["transform"].astype(np.float32).reshape(4, 4)[:, :3]
        first = int(m["indexOffset"])
        p = v[idx[first:first + 3 * int(m["indexCount"])]][:, :3]
        with np.errstate(invalid="ignore", over="ignore"):
            out.append(((c[0] * p[:, :1] + c[1] * p[:, 1:2]) + c[2] * p[:, 2:3]) + c[3])
    return np.concatenate(out).astype(np.float32).reshape(-1, 9)


@pytest.mark.parametrize("flags", [0, abi.NODES_QUANTIZED, abi.BUILD_HOST])
@pytest.mark.parametrize("sizes", [(1,), (3, 300, 1, 255), (64, 0, 1, 0), (0, 5000)])
def test_world_triangles_are_the_host_arithmetic(cuda, sizes, flags):
    """Triangles flattened on the device are, bit for bit, the float32
    arithmetic above, also beside instances without triangles."""
    rng = np.random.default_rng(len(sizes) * 100 + sum(sizes))
    s = Scene()
    for n in sizes:
        v = np.concatenate([_soup(n, "soup").reshape(-1, 3), np.ones((3 * n, 1))], 1).astype(np.float32)
        idx = rng.permutation(3 * n).astype(np.uint32)
        md = ModelData(v, idx, np.tile(np.eye(3, dtype=np.float32), (3 * n, 1, 1)), idx.copy())
        m = np.eye(4)
        m[:3] = rng.normal(size=(3, 4))
        s.add_object(md, m, Material(materialIdx=0))
    a = s.build_arrays()
    dev = reina_rt.DeviceScene(a, flags=flags)
    t = dev.export_bvh()[1].reshape(-1, 3, 4)
    got = np.empty((len(t), 9), np.float32)
    got[t[:, 0, 3].copy().view(np.uint32)] = t[:, :, :3].reshape(-1, 9)
    assert np.array_equal(got.view(np.uint32), _flatten(a).view(np.uint32))
    dev.close()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.0e38])
def test_non_finite_triangle_keeps_the_host_bits(cuda, value):
    tri = np.array([[[0, 0, 0], [1, value, 0], [0, 1, 0]]], np.float32)
    a = _arrays(tri)
    a["instances"][0]["transform"][4] = 2.0    # x += 2 y overflows at 3e38
    got = []
    for flags in (0, abi.BUILD_HOST):
        dev = reina_rt.DeviceScene(a, flags=flags)
        got.append(dev.export_bvh()[1].reshape(3, 4)[:, :3].reshape(1, 9).copy())
        dev.close()
    assert not np.isfinite(got[0]).all()
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    assert np.array_equal(got[0], _flatten(a), equal_nan=True)


def _same_hits(torch, a, b, rays):
    h = [torch.zeros((len(rays), 4), device="cuda") for _ in range(2)]
    for dev, out in zip((a, b), h):
        dev.intersect(rays.data_ptr(), out.data_ptr(), len(rays))
    torch.cuda.synchronize()
    assert torch.equal(h[0].view(torch.int32), h[1].view(torch.int32))
    return h[0]


def _aimed_rays(torch, targets, seed, n=4096):
    """Rays from around the unit cube to the targets, in turn."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = torch.zeros((n, 8), device="cuda")
    r[:, 0:3] = torch.rand((n, 3), device="cuda", generator=g) * 5 - 0.5
    c = torch.from_numpy(np.ascontiguousarray(targets, np.float32)).cuda()[torch.arange(n, device="cuda") % len(targets)]
    r[:, 4:7] = torch.nn.functional.normalize(c - r[:, 0:3], dim=1)
    r[:, 7] = 1e4
    return r


@pytest.mark.parametrize("n", [4, 64, 65, 5000])
@pytest.mark.parametrize("scale", [1e19, 1e25, 1e37])
def test_boxes_whose_area_overflows(cuda, n, scale):
    """No split has a finite cost: leaves of 1..3 triangles all the same, every
    triangle in one of them, and a depth that the traversal stack holds."""
    torch = cuda
    arrays = _arrays(_soup(n, "soup") * scale)
    a, b = reina_rt.DeviceScene(arrays), reina_rt.DeviceScene(arrays, flags=abi.BUILD_HOST)
    for dev in (a, b):
        _check_tree(dev, n)
        assert dev.info().max_depth <= 16
    _same_hits(torch, a, b, _aimed_rays(torch, np.eye(3), n))
    a.close()
    b.close()


@pytest.mark.parametrize("n", [4, 64, 65, 5000])
@pytest.mark.parametrize("far", [1e20, 3e38])
def test_one_huge_triangle_beside_others(cuda, n, far):
    """A triangle whose box area overflows takes no other out of the tree."""
    torch = cuda
    t = _soup(n, "soup")
    t[n // 3, 0] = (far, -far, far)
    arrays = _arrays(t)
    a, b = reina_rt.DeviceScene(arrays), reina_rt.DeviceScene(arrays, flags=abi.BUILD_HOST)
    _check_tree(a, n)
    _check_tree(b, n)
    hits = _same_hits(torch, a, b, _aimed_rays(torch, t[np.arange(n) != n // 3].mean(1), n))
    assert float((hits.view(torch.int32)[:, 1] >= 0).float().mean()) > 0.9
    a.close()
    b.close()


@pytest.mark.parametrize("n", [400, 9000])
@pytest.mark.parametrize("corner", [3e38, -3e38])
def test_infinite_box_beside_the_outermost_triangles(cuda, n, corner):
    """A triangle that reaches to infinity (x = 2^32 times its corner) among
    the 64 triangles furthest out on that side, which one wave partitions: its
    boxes hold them all the same."""
    torch = cuda
    t = _soup(n, "soup").astype(np.float32)
    t[:64, :, 0] += np.copysign(np.float32(20.0), np.float32(corner))
    local = t.copy()
    local[:, :, 0] *= np.float32(2.0 ** -32)
    local[10, 0, 0] = corner
    arrays = _arrays(local)
    arrays["instances"][0]["transform"][0] = 2.0 ** 32
    a, b = reina_rt.DeviceScene(arrays), reina_rt.DeviceScene(arrays, flags=abi.BUILD_HOST)
    _check_tree(a, n)
    _check_tree(b, n)
    hits = _same_hits(torch, a, b, _aimed_rays(torch, np.delete(t[:64], 10, 0).mean(1), n))
    assert float((hits.view(torch.int32)[:, 1] >= 0).float().mean()) > 0.9
    a.close()
    b.close()


# the corners of a triangle that is not finite, on the x axis; an infinity is
# 3e38 under an instance that scales x by 2^32, a NaN reaches every axis. The
# centroid is NaN for three NaN corners and for -inf beside +inf.
NON_FINITE = {"nan": (np.nan,) * 3, "negative_nan": (-np.nan,) * 3, "part_nan": (np.nan, 0.0, 2.0 ** -32),
              "inf": (0.0, 3e38, 2.0 ** -32), "both_inf": (-3e38, 0.0, 3e38), "all_inf": (3e38,) * 3}


@pytest.mark.parametrize("kind", list(NON_FINITE) + ["mixed"])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 33, 64, 65, 129, 5000])
def test_non_finite_triangles_take_no_other_out(cuda, n, kind):
    """Triangles that are not finite beside finite ones, several in one wave's
    sort: every triangle is in one leaf once, and a ray finds the closest
    finite triangle."""
    torch = cuda
    rng = np.random.default_rng(n)
    t = _soup(n, "soup").astype(np.float32)
    bad = np.union1d(np.nonzero(rng.random(n) < (0.4 if n < 200 else 0.01))[0], [n // 2])
    good = np.setdiff1d(np.arange(n), bad)
    local = t.copy()
    local[:, :, 0] *= np.float32(2.0 ** -32)
    for i in bad:
        local[i, :, 0] = NON_FINITE[list(NON_FINITE)[i % len(NON_FINITE)] if kind == "mixed" else kind]
    arrays = _arrays(local)
    arrays["instances"][0]["transform"][0] = 2.0 ** 32
    dev = reina_rt.DeviceScene(arrays)
    nodes, tris = dev.export_bvh()
    tris = tris.reshape(-1, 3, 4)
    assert np.array_equal(np.sort(tris[:, 0, 3].copy().view(np.uint32)), np.arange(n))
    assert np.isfinite(tris[:, :, :3]).all((1, 2)).sum() == len(good)
    nodes = nodes.reshape(-1, 256)
    first = (nodes[:, 196:200].copy().view(np.uint32) & 0xFFFFFF).astype(int)
    meta = nodes[:, 200:208].astype(int)
    leaf = (meta != 0) & (meta < 0x80)
    slots = [(first + (meta & 31) + j)[leaf & ((meta >> 5) > j)] for j in range(3)]
    assert np.array_equal(np.sort(np.concatenate(slots)), np.arange(n))
    if len(good) == 0:
        dev.close()
        return
    ref = reina_rt.DeviceScene(_arrays(t[good]))
    rays = _aimed_rays(torch, t[good].mean(1), n)
    h, hr = torch.zeros((4096, 4), device="cuda"), torch.zeros((4096, 4), device="cuda")
    dev.intersect(rays.data_ptr(), h.data_ptr(), 4096)
    ref.intersect(rays.data_ptr(), hr.data_ptr(), 4096)
    torch.cuda.synchronize()
    prim, pref = (x.view(torch.int32)[:, 1].cpu().numpy() for x in (h, hr))
    assert (pref >= 0).mean() > 0.9
    assert np.array_equal(prim, np.where(pref >= 0, good[np.maximum(pref, 0)], -1))
    assert torch.equal(h[:, 0].view(torch.int32), hr[:, 0].view(torch.int32))
    dev.close()
    ref.close()
