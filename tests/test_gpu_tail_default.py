"""Where a frame starts by default: up to 2^22 paths in the tail launch, beyond
that, with next-event estimation, or when the extend kernel is counted or
timed, in bounce iterations. The image does not depend on it."""
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
    assert dev.get_tuning()["tail_paths"] == 1 << 20
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
