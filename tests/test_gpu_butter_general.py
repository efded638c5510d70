"""Butteraugli pairs beyond the matrix-core strips' range (float samples above
linear 32, opsin values above 8,192), which the general kernels
(vship_amd/csrc/butter.hip) score, against the FP64 oracle: norms and maps on
sizes at the edges of their tiles, several such pairs in one batch, and what
they cost beside an ordinary pair.

The values are chosen so that strips could not represent them: 12 is linear
389, stored times 1,024, and fp16 ends at 65,504."""
import time

import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests import butter_lib as bl
from tests.gpu_helpers import rgb_pair, say

pytestmark = pytest.mark.gpu

# The bounds of the other Butteraugli tests. The metric in FP32 on a CPU, with
# these samples, is within 2e-6 (norms) and 2e-5 (maps) of 64 bits.
NORM_RTOL = 1e-4
MAP_RTOL, MAP_ATOL = 1e-4, 1e-6


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


def far_pair(w, h, seed, value=12.0, fmt=api.PF_RGB_F32):
    ref, dist = rgb_pair(w, h, fmt, seed)
    dist[1][h // 2, w // 3] = value
    return ref, dist


def checkered_pair(w, h, seed):
    """Samples of +-3 (linear 14) whose blur is near 0: the opsin gain of a dark
    surround times a bright sample, 40,000 at intensity 203."""
    ref, dist = rgb_pair(w, h, api.PF_RGB_F32, seed)
    yy, xx = np.mgrid[0:h, 0:w]
    board = np.where((yy + xx) % 2, 3.0, -3.0).astype(np.float32)
    for p in dist:
        p[h // 4:h // 2, w // 4:w // 2] = board[h // 4:h // 2, w // 4:w // 2]
    return ref, dist


def norms_and_maps(pairs, qnorm=2, fmt=api.PF_RGB_F32):
    h, w = pairs[0][0][0].shape
    dp = api.ButterDevicePairs(pairs, distmaps=True, fmt=fmt)
    try:
        with api.ButteraugliBatch(w, h, len(pairs), qnorm) as b:
            return b.compute(dp), [dp.distmap(i) for i in range(len(pairs))]
    finally:
        dp.free()


def check(norms, gmap, pair, qnorm=2):
    want, wmap = bl.butteraugli(*[[p.astype(np.float32) for p in im] for im in pair], qnorm, diffmap=True)
    say(f"  norms {np.abs(norms / want - 1).max():.1e} map {np.max(np.abs(gmap - wmap) / np.abs(wmap)):.1e}")
    assert np.all(np.abs(norms - want) <= NORM_RTOL * np.abs(want))
    assert np.all(np.abs(gmap - wmap) <= MAP_ATOL + MAP_RTOL * np.abs(wmap))


# on and one past the general kernels' tiles (blurs 64 x 32, Malta 64 x 16), at
# both scales, and narrower than the widest window
@pytest.mark.parametrize("w,h", [(1, 1), (7, 5), (20, 130), (64, 32), (65, 33), (127, 31), (129, 17), (130, 97)])
@pytest.mark.parametrize("value", [12.0, -12.0])
def test_far_samples(w, h, value):
    say(f"case far sample {value} {w}x{h}")
    pair = far_pair(w, h, 100 * w + h, value)
    norms, maps = norms_and_maps([pair])
    check(norms[0], maps[0], pair)


def test_far_half_samples():
    say("case far samples, half floats, 3-norm")
    pair = far_pair(70, 50, 5, 15.0, api.PF_RGB_F16)
    norms, maps = norms_and_maps([pair], 3, api.PF_RGB_F16)
    check(norms[0], maps[0], pair, 3)


def test_far_opsin_values():
    say("case far opsin values")
    pair = checkered_pair(96, 80, 5)
    norms, maps = norms_and_maps([pair])
    check(norms[0], maps[0], pair)


@pytest.mark.parametrize("largest", [12.0, 1e15], ids=["scaled", "unscaled"])
def test_several_far_pairs(largest):
    """Far pairs between ordinary ones score as alone, and so do the ordinary
    ones, also where one far pair's linear values (1e15: 1e36) have no room for
    the strips' factor in FP32."""
    say(f"case several far pairs, up to {largest}")
    w, h = 75, 60
    pairs = [rgb_pair(w, h, api.PF_RGB_F32, 1), far_pair(w, h, 2), rgb_pair(w, h, api.PF_RGB_F32, 3),
             checkered_pair(w, h, 4), far_pair(w, h, 5, largest), rgb_pair(w, h, api.PF_RGB_F32, 6)]
    norms, maps = norms_and_maps(pairs)
    for i, p in enumerate(pairs):
        alone, amap = norms_and_maps([p])
        assert np.array_equal(norms[i], alone[0], equal_nan=True)
        assert np.array_equal(maps[i], amap[0], equal_nan=True)
    for i in (0, 1, 2, 3, 5):
        check(norms[i], maps[i], pairs[i])


def test_the_strips_leave_far_pairs_out():
    """The general kernels alone take 1.5 times the strips' time; with the strips'
    before them it was 2.5."""
    say("case time of far pairs")
    w, h, n = 1920, 1080, 8
    plain = [rgb_pair(w, h, api.PF_RGB_F32, 1)] * n
    far = [far_pair(w, h, 1)] * n
    best = []
    for pairs in (plain, far):
        dp = api.ButterDevicePairs(pairs)
        with api.ButteraugliBatch(w, h, n) as b:
            b.compute(dp)
            t = []
            for _ in range(20):
                t0 = time.perf_counter()
                b.compute(dp)
                t.append(time.perf_counter() - t0)
        dp.free()
        best.append(min(t))
    say(f"  {best[0] * 1e6:.0f} us, far pairs {best[1] * 1e6:.0f} us")
    assert best[1] < 2.0 * best[0]


@pytest.mark.parametrize("fmt", [api.PF_RGB_F32, api.PF_RGB_F16])
def test_nan_samples_count_as_zero(fmt):
    """A NaN sample linearises to 0, in the strips' range like any other."""
    say("case NaN sample")
    nan, zero = (norms_and_maps([far_pair(70, 50, 5, v, fmt)], 2, fmt) for v in (np.nan, 0.0))
    assert np.isfinite(zero[0]).all()
    assert np.array_equal(nan[0], zero[0])
    assert np.array_equal(nan[1][0], zero[1][0])
