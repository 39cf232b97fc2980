"""The shading kernels' shortcuts against what they stand for: roots and
inverses, whole numbers over 255, texel indices without an integer division, the tangent frame left
out where no surface reads it."""
import numpy as np
import pytest

import oracle
import reina_rt
from reina_rt import scenes
from reina_rt.scene import make_desc


@pytest.mark.gpu
def test_texel_bytes_over_255_are_the_rounded_quotients(cuda):
    """The device function for every byte, bit for bit."""
    torch = cuda
    n = torch.arange(256, device="cuda", dtype=torch.float32)
    out = torch.zeros_like(n)
    reina_rt.debug_math(9, n.data_ptr(), None, out.data_ptr(), 256)
    torch.cuda.synchronize()
    want = np.arange(256, dtype=np.float32) / np.float32(255.0)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_over_255_is_the_rounded_quotient():
    """Why the shortcut is exact: n * c corrected by its exact remainder equals n / 255 for every texel
    value (products of two float32 are exact in float64, so each fused
    multiply-add is one float64 expression rounded once)."""
    n = np.arange(256, dtype=np.float32)
    c = np.float32(1.0) / np.float32(255.0)
    q = n * c
    r = (np.float64(-255.0) * q.astype(np.float64) + n).astype(np.float32)
    got = (r.astype(np.float64) * np.float64(c) + q).astype(np.float32)
    assert np.array_equal(got, n / np.float32(255.0))


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (257, 2)])
def test_texture_sizes_equal_oracle(cuda, w, h):
    """Odd texture sizes on every map: the bump search at grazing angles walks
    many textures away, past what one wrap brings back. Lambertian walls
    without maps and mapped ones lie in one frame, so waves mix surfaces with
    and without a tangent frame."""
    torch = cuda
    sc, _ = scenes.textured_cornell()
    arrays = sc.build_arrays()
    rng = np.random.default_rng(w * 100 + h)
    arrays["textures"] = [rng.integers(0, 256, (h, w, 4), dtype=np.uint8) for _ in arrays["textures"]]
    W, H = 40, 36
    pc = scenes.cornell_push(W, H, spp=3, max_bounces=6)
    dev = reina_rt.DeviceScene(arrays)
    img = torch.zeros((H, W, 4), device="cuda")
    dev.trace(pc, img.data_ptr(), W, H)
    torch.cuda.synchronize()
    ref, _ = oracle.OracleScene(arrays, make_desc).render(pc, W, H, use_bvh=False)
    got = img.cpu().numpy()
    assert ((got.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(got) & np.isnan(ref))).all()
    dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [4, 7, 8], ids=["sqrt", "inverse", "inverse_sqrt"])
def test_root_and_inverse_are_correctly_rounded(cuda, fn):
    """sqrt, 1 / x and 1 / sqrt(x) against IEEE arithmetic on the host: every
    mantissa of two neighbouring binades, every exponent, and the inputs
    around the ends of the short forms' ranges."""
    torch = cuda
    man = np.arange(1 << 24, dtype=np.uint32) + np.uint32(0x3F800000)          # [1, 4)
    exps = ((np.arange(256, dtype=np.uint32) << 23)[:, None] |
            np.array([0, 1, 2, 0x2AAAAA, 0x3FFFFF, 0x400000, 0x7FFFFE, 0x7FFFFF], np.uint32)[None]).reshape(-1)
    edge = (np.array([0x0D800000, 0x7E800000, 0x01800000, 0x7E000000], np.uint32)[:, None] +
            np.arange(-8, 9).astype(np.uint32)[None]).reshape(-1)
    bits = np.concatenate([man, exps, edge, exps | np.uint32(0x80000000), edge | np.uint32(0x80000000)])
    x = bits.view(np.float32)
    with np.errstate(all="ignore"):
        ref = {4: np.sqrt(x), 7: np.float32(1.0) / x, 8: np.float32(1.0) / np.sqrt(x)}[fn]
    t = torch.from_numpy(x.copy()).cuda()
    out = torch.zeros_like(t)
    reina_rt.debug_math(fn, t.data_ptr(), None, out.data_ptr(), len(x))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    same = (got.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(got) & np.isnan(ref))
    assert same.all(), [hex(b) for b in bits[~same][:8]]


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [4, 7, 8], ids=["sqrt", "inverse", "inverse_sqrt"])
def test_root_and_inverse_of_every_float(cuda, fn):
    """All 2^32 inputs against double precision rounded to float. The double
    result has more than 2 x 24 + 1 bits, so rounding it again is the correctly
    rounded root or quotient; 1 / sqrt(x) rounds both steps."""
    torch = cuda
    step = 1 << 26
    out = torch.empty(step, device="cuda")
    bad = 0
    for start in range(-(1 << 31), 1 << 31, step):
        x = torch.arange(start, start + step, device="cuda", dtype=torch.int64).to(torch.int32).view(torch.float32)
        reina_rt.debug_math(fn, x.data_ptr(), None, out.data_ptr(), step,
                            stream=torch.cuda.current_stream().cuda_stream)
        d = x.double()
        if fn == 4:
            ref = d.sqrt().float()
        elif fn == 7:
            ref = d.reciprocal().float()
        else:
            ref = d.sqrt().float().double().reciprocal().float()
        same = (out.view(torch.int32) == ref.view(torch.int32)) | (torch.isnan(out) & torch.isnan(ref))
        bad += int((~same).sum())
    assert bad == 0
