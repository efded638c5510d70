"""Butteraugli's matrix-core strips (vship_amd/csrc/butter_strip.hip) against
the FP64 oracle where they can go wrong: sizes on and one past the strips'
blocks (32 columns in two halves of 16, rows in blocks of 16, strips of 16 to
256 rows) and smaller than the widest window, and pairs whose samples lie
beyond the strips' range, which the general kernels score instead."""
import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests import butter_lib as bl
from tests.gpu_helpers import rgb_pair, say

pytestmark = pytest.mark.gpu

# the bounds of the other Butteraugli tests (FP32 arithmetic against FP64)
NORM_RTOL = 1e-4
MAP_RTOL, MAP_ATOL = 1e-4, 1e-6


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


def norms_and_maps(pairs):
    h, w = pairs[0][0][0].shape
    dp = api.ButterDevicePairs(pairs, distmaps=True)
    try:
        with api.ButteraugliBatch(w, h, len(pairs)) as b:
            return b.compute(dp), [dp.distmap(i) for i in range(len(pairs))]
    finally:
        dp.free()


@pytest.mark.parametrize("w,h", [(16, 16), (17, 33), (31, 129), (32, 31), (33, 15), (47, 48), (65, 257), (200, 9)])
def test_strip_edges(w, h):
    say(f"case strip edges {w}x{h}")
    ref, dist = rgb_pair(w, h, api.PF_RGB_F32, 100 * w + h)
    (got,), (gmap,) = norms_and_maps([(ref, dist)])
    want, wmap = bl.butteraugli(ref, dist, diffmap=True)
    assert np.all(np.abs(got - want) <= NORM_RTOL * np.abs(want))
    assert np.all(np.abs(gmap - wmap) <= MAP_ATOL + MAP_RTOL * np.abs(wmap))


@pytest.mark.parametrize("value", [4.3, -4.3, np.inf])
def test_values_beyond_the_strips_range(value):
    """4.3 is linear 33, just beyond the range of 32; the difference it makes
    dominates the norms, whose FP32 error is then far below the bound. The
    pairs beside it score as they do alone."""
    w, h = 96, 80
    say(f"case beyond the range: {value}")
    plain = [rgb_pair(w, h, api.PF_RGB_F32, s) for s in (1, 2)]
    ref, dist = rgb_pair(w, h, api.PF_RGB_F32, 3)
    dist[1][40, 50] = value
    alone = [norms_and_maps([p]) for p in (plain[0], (ref, dist), plain[1])]
    norms, maps = norms_and_maps([plain[0], (ref, dist), plain[1]])
    for i in range(3):
        assert np.array_equal(norms[i], alone[i][0][0], equal_nan=True)
        assert np.array_equal(maps[i], alone[i][1][0], equal_nan=True)
    if np.isfinite(value):
        want = bl.butteraugli(ref, dist)
        assert np.all(np.abs(norms[1] - want) <= NORM_RTOL * np.abs(want))
    assert np.isfinite(norms[[0, 2]]).all()
