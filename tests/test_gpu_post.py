"""Bloom and tone mapping: the per-row and per-column kernels (and the kernels
that take the sizes those do not) equal the oracle's restatement bit for bit
over sizes at the edges of their tiles, radii and non-finite samples."""
import numpy as np
import pytest

import oracle
import reina_rt

pytestmark = pytest.mark.gpu


def _check(torch, img, radius, threshold):
    H, W = img.shape[:2]
    ref_out, ref_comb = oracle.postprocess(img, radius=radius, threshold=threshold, intensity=0.25, exposure=0.5)
    t_in = torch.from_numpy(img).cuda()
    scratch = torch.full((2, H, W, 4), float("nan"), device="cuda")
    out = torch.zeros((H, W, 4), dtype=torch.uint8, device="cuda")
    reina_rt.postprocess(t_in.data_ptr(), scratch.data_ptr(), out.data_ptr(), W, H, radius, threshold, 0.25, 0.5)
    torch.cuda.synchronize()
    comb = scratch[0].cpu().numpy()
    same = (comb.view(np.uint32) == ref_comb.view(np.uint32)) | (np.isnan(comb) & np.isnan(ref_comb))
    assert same.all()
    assert np.array_equal(out.cpu().numpy(), ref_out)


# radius 5: half-widths k from 0 (4 pixels and fewer) past the last tap with a
# weight (72: images over 480 pixels); 40 on 500 pixels: more taps than the
# kernel arguments hold; 5300 and 5500 pixels at radius 1: the longest rows that
# fit the 64 KB stage (64,176 bytes) and past it
@pytest.mark.parametrize("W,H,radius", [(1, 1, 5.0), (3, 2, 5.0), (63, 5, 5.0), (64, 9, 5.0), (65, 33, 0.7),
                                        (257, 31, 5.0), (487, 3, 5.0), (1023, 513, 5.0), (1030, 521, 2.0), (60, 700, 5.0),
                                        (500, 7, 40.0), (5300, 3, 1.0), (5500, 3, 1.0)])
def test_postprocess_sizes_bitexact(cuda, W, H, radius):
    rng = np.random.default_rng(W * 1000 + H)
    img = (rng.random((H, W, 4)) ** 4 * 4.0 - 0.1).astype(np.float32)
    img[..., 3] = 1.0
    _check(cuda, img, radius, 1.0)


# 700 x 800 takes several outputs per lane, 600 x 90 one
@pytest.mark.parametrize("W,H", [(700, 800), (600, 90)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3.0e38])
def test_postprocess_non_finite_bitexact(cuda, W, H, value):
    """A sample that is not finite reaches every pixel within the stencil's
    half-width, also where its weight is zero (0 * inf and 0 * NaN are NaN)."""
    rng = np.random.default_rng(5)
    img = rng.random((H, W, 4)).astype(np.float32)
    img[H // 3, W // 4, 1] = value
    img[H // 3, W // 4 + 1, 0] = value
    _check(cuda, img, 5.0, 0.5)


# half-widths below, at and past the last tap with a weight (k 0, 1, 9, 72, 75,
# 162), where the weighted taps are rounded up past the stencil's end, one and
# several outputs per lane, samples at the corners and all over
@pytest.mark.parametrize("W,H,radius", [(1, 1, 5.0), (9, 7, 5.0), (60, 61, 5.0), (64, 70, 0.7), (487, 3, 5.0), (3, 487, 5.0),
                                        (500, 500, 5.0), (601, 90, 2.0), (730, 725, 5.0), (1100, 500, 5.0),
                                        (480, 1100, 5.0), (300, 420, 20.0)])
@pytest.mark.parametrize("where", ["corners", "all"])
def test_postprocess_non_finite_sizes_bitexact(cuda, W, H, radius, where):
    rng = np.random.default_rng(W * 1000 + H)
    img = rng.random((H, W, 4)).astype(np.float32)
    values = np.array([np.nan, np.inf, -np.inf, 3.0e38, 2.0e34, -3.0e38], np.float32)
    if where == "corners":
        for n, (y, x) in enumerate(((0, 0), (0, W - 1), (H - 1, 0), (H - 1, W - 1))):
            img[y, x, n % 3] = values[n]
    else:
        bad = rng.random((H, W, 3)) < 3.0 / max(W, H)
        img[..., :3][bad] = rng.choice(values, int(bad.sum()))
    _check(cuda, img, radius, 0.5)


def test_non_finite_samples_cost_a_few_times_finite_ones(cuda):
    """Every tap of every pixel (2k + 1 = 325 and 407 at 1080 x 1350) instead
    of the 145 with a weight: about twice the time (it was 17 times while each
    output loaded its own samples)."""
    torch = cuda
    W, H = 1080, 1350
    out = torch.zeros((H, W, 4), dtype=torch.uint8, device="cuda")
    scratch = torch.zeros((2, H, W, 4), device="cuda")
    img = torch.rand((H, W, 4), device="cuda")
    bad = img.clone()
    bad[:, W // 3, 0] = float("nan")
    ms = []
    for x in (img, bad):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        t = []
        for _ in range(9):
            e[0].record()
            reina_rt.postprocess(x.data_ptr(), scratch.data_ptr(), out.data_ptr(), W, H, 5.0, 0.5, 0.25, 0.5,
                                 stream=torch.cuda.current_stream().cuda_stream)
            e[1].record()
            torch.cuda.synchronize()
            t.append(e[0].elapsed_time(e[1]))
        ms.append(sorted(t)[4])
    assert ms[1] < 8 * ms[0], ms
