"""Closest-hit queries on either side of the batch size where the queue kernel
takes over (2^18 rays): every ray once, the same hits and per-ray counters,
for partial waves, FP32 and 8-bit nodes, and any launch shape of the queue."""
import numpy as np
import pytest

import reina_rt
from reina_rt import abi, scenes

pytestmark = pytest.mark.gpu

LIMIT = 1 << 18


@pytest.fixture(scope="module")
def arrays():
    return scenes.icosphere(levels=4)[0].build_arrays()


def _rays(torch, n):
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    r = torch.zeros((n, 8), device="cuda")
    r[:, 0:3] = torch.rand((n, 3), device="cuda", generator=g) * 3 - 1.5
    r[:, 4:7] = torch.nn.functional.normalize(torch.randn((n, 3), device="cuda", generator=g), dim=1)
    r[:, 7] = 1e4
    r[7, 4:7] = 0.0            # no direction: a miss
    r[11, 0] = float("nan")
    return r


def _query(torch, dev, rays, count=False, noalloc=False):
    n = len(rays)
    hits = torch.full((n + 1, 4), -7.0, device="cuda")
    cnt = torch.full((n + 1, 2), -7, dtype=torch.int32, device="cuda") if count else None
    if noalloc:
        reina_rt.check(reina_rt.lib().reina_rt_intersect_noalloc(dev.handle, rays.data_ptr(), hits.data_ptr(), n, None))
    else:
        dev.intersect(rays.data_ptr(), hits.data_ptr(), n, cnt.data_ptr() if count else None)
    torch.cuda.synchronize()
    assert (hits[n] == -7.0).all()         # nothing past the end
    return hits[:n].view(torch.int32), (cnt[:n] if count else None)


@pytest.mark.parametrize("flags", [0, abi.NODES_QUANTIZED], ids=["fp32", "q8"])
def test_batches_around_the_limit(cuda, arrays, flags):
    torch = cuda
    dev = reina_rt.DeviceScene(arrays, flags=flags)
    rays = _rays(torch, LIMIT + 70001)
    parts = [_query(torch, dev, rays[a:a + LIMIT], count=True) for a in (0, LIMIT)]
    hits, cnt = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
    assert int((hits[:, 1] >= 0).sum()) > 10000
    # partial waves of every spread (4, 8, 16, 32 and 64 rays per wave)
    for n in (1, 3, 4, 5, 8191, 8193, 16385, 32769, 65537, LIMIT - 1):
        h, c = _query(torch, dev, rays[:n], count=n % 2 == 1)
        assert torch.equal(h, hits[:n]), n
        assert c is None or torch.equal(c, cnt[:n])
    # the queue: partition ends that claims meet exactly or run past
    for grid, claim in ((1, 64), (8, 512), (256, 128), (2048, 64), (4096, 512)):
        dev.set_tuning(grid_blocks=grid, claim_rays=claim)
        for n in (LIMIT + 1, LIMIT + 8 * 512 + 3, LIMIT + 70001) if grid > 8 else (LIMIT + 8 * 512 + 3,):
            h, c = _query(torch, dev, rays[:n], count=grid == 256)
            assert torch.equal(h, hits[:n]), (grid, claim, n)
            assert c is None or torch.equal(c, cnt[:n])
    for n in (5, LIMIT, LIMIT + 1, LIMIT + 70001):
        assert torch.equal(_query(torch, dev, rays[:n], noalloc=True)[0], hits[:n]), n
    dev.close()


@pytest.mark.parametrize("flags", [0, abi.NODES_QUANTIZED], ids=["fp32", "q8"])
def test_every_stack_depth(cuda, arrays, flags):
    """The kernels of each LDS stack size on both sides of the limit, plain and
    counting; at 24 and 32 entries fewer blocks are resident than 2^18 rays
    launch."""
    torch = cuda
    dev = reina_rt.DeviceScene(arrays, flags=flags)
    rays = _rays(torch, LIMIT + 70001)
    hits, cnt = _query(torch, dev, rays, count=True)
    for depth in (8, 16, 24, 32):
        dev.set_tuning(stack_depth=depth)
        for n in (1000, LIMIT, LIMIT + 70001):
            for count in (False, True):
                h, c = _query(torch, dev, rays[:n], count=count)
                assert torch.equal(h, hits[:n]), (depth, n)
                assert c is None or torch.equal(c, cnt[:n]), (depth, n)
    dev.close()


@pytest.mark.parametrize("n", [1000, LIMIT + 9])
def test_noalloc_replays_in_a_graph(cuda, arrays, n):
    """Both kernels under capture, replayed with eager work between."""
    torch = cuda
    dev = reina_rt.DeviceScene(arrays)
    rays = _rays(torch, n)
    ref, _ = _query(torch, dev, rays)
    hits = torch.zeros((n, 4), device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        reina_rt.check(reina_rt.lib().reina_rt_intersect_noalloc(dev.handle, rays.data_ptr(), hits.data_ptr(), n,
                                                                 torch.cuda.current_stream().cuda_stream))
    for _ in range(3):
        hits.zero_()
        _query(torch, dev, rays)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(hits.view(torch.int32), ref)
    dev.close()
