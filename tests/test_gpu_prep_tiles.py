"""The convert/pyramid kernel's tiles of 128 x 32 at sizes that end on, one
before or one past a tile, for the staged 4:2:0 path and every RGB format,
against the FP64 oracle; and the same scores bit for bit from planes that start
one sample past an aligned address with rows of an odd number of samples (the
samples of a whole tile are loaded two at a time)."""
import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests import oracle_lib as ol
from tests.gpu_helpers import gpu_batch, oracle_rgb, rgb_pair, say

pytestmark = pytest.mark.gpu

SCORE_ATOL = 1e-3  # the bar of every score against the oracle
SIZES = [(128, 32), (127, 33), (129, 31), (256, 64), (257, 65), (255, 96)]
FORMATS = [(api.PF_YUV420_U8, 8), (api.PF_YUV420_U16, 10), (api.PF_RGB_U8, 0), (api.PF_RGB_U16, 0), (api.PF_RGB_F16, 0),
           (api.PF_RGB_F32, 0)]


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


def frames(w, h, fmt, bits):
    if not bits:
        return rgb_pair(w, h, fmt, 5 * w + h)
    f, g = rgb_pair(w, h, api.PF_RGB_F32, 5 * w + h)
    s, dt = 1 << (bits - 8), np.uint8 if bits == 8 else np.uint16

    def yuv(x):
        return [np.round(16 * s + r * s * p.astype(np.float64)).astype(dt)
                for r, p in ((219, x[0]), (224, x[1][::2, ::2]), (224, x[2][::2, ::2]))]

    return yuv(f), yuv(g)


@pytest.mark.parametrize("fmt,bits", FORMATS)
@pytest.mark.parametrize("w,h", SIZES)
def test_tiles_and_alignment(w, h, fmt, bits):
    say(f"case prep tiles {w}x{h} format {fmt}")
    ref, dist = frames(w, h, fmt, bits)
    (got,), feats = gpu_batch([(ref, dist)], fmt, bits=bits or 8)
    if bits:
        want, _ = ol.score_yuv420(ref, dist, bits, ol.SO_MAT_BT709)
    else:
        want, _ = oracle_rgb(ref, dist, fmt)
    assert abs(got - want) <= SCORE_ATOL
    # the same planes, one sample past an aligned address, in rows of an odd number of samples
    size = ref[0].itemsize
    plane = (((w | 1) + 2) * (h + 1) * size + 255) // 256 * 256
    buf = api.DeviceBuffer(6 * plane)
    desc = (api.Pair * 1)()
    d = desc[0]
    for k, p in enumerate(ref + dist):
        n = (p.shape[1] | 1) + 2
        wide = np.zeros((p.shape[0], n), p.dtype)
        wide[:, :p.shape[1]] = p
        buf.upload(wide, k * plane + size)
        (d.ref if k < 3 else d.dist)[k % 3] = buf.ptr + k * plane + size
        (d.ref_stride if k < 3 else d.dist_stride)[k % 3] = n * size
    d.width, d.height, d.format, d.bits, d.matrix, d.chroma_location = w, h, fmt, bits or 8, api.MATRIX_BT709, api.CHROMA_LEFT
    with api.SSIMU2Batch(1, w, h) as b:
        s, f = b.compute(desc, features=True)
    buf.free()
    assert s[0] == got and np.array_equal(f, feats)


@pytest.mark.parametrize("layout,bits,loc", [("444", 8, api.CHROMA_LEFT), ("444", 10, api.CHROMA_CENTER),
                                             ("422", 8, api.CHROMA_LEFT), ("422", 10, api.CHROMA_TOPLEFT),
                                             ("422", 16, api.CHROMA_LEFT), ("422", 8, api.CHROMA_CENTER)])
@pytest.mark.parametrize("w,h", [(257, 32), (384, 64), (387, 65), (518, 97)])
def test_layouts_of_whole_tiles(w, h, layout, bits, loc):
    """Whole tiles of 4:4:4 and left-located 4:2:2 load their chroma directly; the tiles at the picture's sides,
    and every other layout, form each sample's position and weights."""
    f8, f16, sw, sh = api.YUV_LAYOUTS[layout]
    say(f"case prep layouts {w}x{h} YUV{layout} {bits}-bit location {loc}")
    rng = np.random.default_rng(w + h + bits)
    s, dt = 1 << (bits - 8), np.uint8 if bits == 8 else np.uint16
    f, _ = rgb_pair(w, h, api.PF_RGB_F32, w + bits)
    sub = (slice(None, None, 1 << sh), slice(None, None, 1 << sw))
    ref = [np.round(16 * s + r * s * p.astype(np.float64)).astype(dt)
           for r, p in ((219, f[0]), (224, f[1][sub]), (224, f[2][sub]))]
    # (codes beyond a 10-bit depth are clamped to it)
    dist = [np.clip(np.round(p + 3 * s * rng.standard_normal(p.shape)), 0, (1 << bits) - 1 + (bits == 10) * 3).astype(dt)
            for p in ref]
    want, fo = ol.score_yuv(ref, dist, bits, ol.SO_MAT_BT709, sw, sh, loc)
    (got,), feats = gpu_batch([(ref, dist)], f8 if bits == 8 else f16, bits=bits, chroma_location=loc)
    assert abs(got - want) <= SCORE_ATOL
    assert np.all(np.abs(feats[0] - fo) <= 2e-5 + 1e-3 * np.abs(fo))
