"""Where a frame starts by default: up to 2^22 paths in the tail launch, beyond
that, with next-event estimation, or when the extend kernel is counted or
timed, in bounce iterations. A threshold that the caller sets is taken as it
is, 2^20 among them. The image does not depend on it."""
import pytest

import reina_rt
from reina_rt import abi, scenes
from reina_rt.scene import push_consts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,options,whole", [(1025, 1024, 0, True), (2048, 2048, 0, True), (2049, 2048, 0, False),
                                               (1025, 1024, abi.TRACE_NEE, False), (1025, 1024, abi.TRACE_COUNT, False),
                                               (1025, 1024, abi.TRACE_TIME_EXTEND, False),
                                               (1024, 1024, abi.TRACE_NEE, True)])
def test_default_tail_paths(cuda, W, H, options, whole):
    torch = cuda
    scene, cam = scenes.cornell()
    dev = reina_rt.DeviceScene(scene.build_arrays())
    assert dev.get_tuning()["tail_paths"] == abi.TAIL_AUTO
    dev.set_trace_options(options)
    pc = push_consts(cam["eye"], cam["center"], cam["fov"], W, H, 2, 3)
    img = [torch.zeros((H, W, 4), device="cuda") for _ in range(2)]
    dev.trace(pc, img[0].data_ptr(), W, H)
    st = dev.stats()
    assert (st.tail_rays == st.extension_rays) == whole
    dev.set_tuning(tail_paths=0)
    dev.trace(pc, img[1].data_ptr(), W, H)
    assert dev.stats().extension_rays == st.extension_rays and dev.stats().tail_rays == 0
    assert torch.equal(img[0], img[1])
    dev.close()


@pytest.mark.parametrize("tail,whole", [((1 << 20) - 1, False), (1 << 20, False), ((1 << 20) + 1024, True),
                                        (1 << 22, True), (abi.TAIL_OFF, True), (abi.TAIL_AUTO, True), (0, False)])
def test_tail_paths_as_set(cuda, tail, whole):
    """1025 x 1024 = 2^20 + 1024 paths: thresholds around 2^20 as numbers."""
    torch = cuda
    W, H = 1025, 1024
    scene, cam = scenes.cornell()
    dev = reina_rt.DeviceScene(scene.build_arrays())
    dev.set_tuning(tail_paths=tail)
    dev.set_tuning(refill_min=16)
    assert dev.get_tuning()["tail_paths"] == tail        # kept by a call that sets another field
    img = torch.zeros((H, W, 4), device="cuda")
    dev.trace(push_consts(cam["eye"], cam["center"], cam["fov"], W, H, 2, 3), img.data_ptr(), W, H)
    st = dev.stats()
    assert (st.tail_rays == st.extension_rays) == whole
    dev.set_tuning(**dict(dev.get_tuning(), tail_paths=abi.TAIL_AUTO))
    dev.trace(push_consts(cam["eye"], cam["center"], cam["fov"], W, H, 2, 3), img.data_ptr(), W, H)
    assert dev.stats().tail_rays == dev.stats().extension_rays
    dev.close()


@pytest.mark.parametrize("flags", [0, abi.NODES_QUANTIZED], ids=["fp32", "q8"])
@pytest.mark.parametrize("nee", [False, True], ids=["plain", "nee"])
def test_tail_at_every_stack_depth(cuda, flags, nee):
    """The tail kernel of each LDS stack size, on grids that fit the GPU at
    once (256 x 256: 256 blocks) and that do not (640 x 480: 1,200), against
    bounce iterations."""
    torch = cuda
    scene, cam = scenes.icosphere(levels=3)
    dev = reina_rt.DeviceScene(scene.build_arrays(), flags=flags)
    dev.set_trace_options(abi.TRACE_NEE if nee else 0)
    for W, H in ((256, 256), (640, 480)):
        pc = push_consts(cam["eye"], cam["center"], cam["fov"], W, H, 2, 6)
        ref, img = (torch.zeros((H, W, 4), device="cuda") for _ in range(2))
        dev.set_tuning(tail_paths=0)
        dev.trace(pc, ref.data_ptr(), W, H)
        rays = dev.stats().extension_rays
        for depth in (8, 16, 24, 32):
            dev.set_tuning(tail_paths=1 << 30, stack_depth=depth)
            img.zero_()
            dev.trace(pc, img.data_ptr(), W, H)
            st = dev.stats()
            assert st.tail_rays == st.extension_rays == rays
            assert torch.equal(img.view(torch.int32), ref.view(torch.int32)), (W, depth)
    dev.close()
