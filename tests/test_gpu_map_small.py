"""The FP64 map tiles of 16 x 16 (vship_amd/csrc/map_small.hpp) against the
FP64 oracle on sizes whose segments end on, one before or one past a tile, are
one pixel wide, or lie on either side of the 4,096-pixel line to the matrix
cores; and the same scores bit for bit whether the tiles ride along with the
matrix-core launch (eager), or are launched by themselves (persistent grid,
captured graph)."""
import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests.gpu_helpers import gpu_batch, oracle_rgb, rgb_pair, say

pytestmark = pytest.mark.gpu

SCORE_ATOL = 1e-3  # the bar of every score against the oracle
SIZES = [(16, 16), (17, 15), (33, 31), (64, 63), (64, 64), (65, 64), (1, 300), (300, 1), (95, 47), (130, 127)]


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


@pytest.mark.parametrize("fmt", [api.PF_RGB_U8, api.PF_RGB_F32])
@pytest.mark.parametrize("w,h", SIZES)
def test_small_segments(w, h, fmt):
    say(f"case small segments {w}x{h} format {fmt}")
    ref, dist = rgb_pair(w, h, fmt, 7 * w + h)
    want, _ = oracle_rgb(ref, dist, fmt)
    (got,), feats = gpu_batch([(ref, dist)], fmt, th=api_mfma())
    assert abs(got - want) <= SCORE_ATOL
    for kw in (dict(persistent_grid=7), dict(persistent_grid=512, graph=True)):
        (other,), of = gpu_batch([(ref, dist)], fmt, th=api_mfma(), **kw)
        assert other == got and np.array_equal(of, feats), kw


def api_mfma():
    return 1  # VSHIP_MAP_MFMA


def test_batch_of_small_frames_equals_each_alone():
    """Float and integer frames take different map groups; the FP64 tiles of all go with one launch."""
    say("case batch of small frames")
    pairs = [rgb_pair(w, h, api.PF_RGB_U8, i) for i, (w, h) in enumerate(SIZES)]
    scores, feats = gpu_batch(pairs, api.PF_RGB_U8)
    for i, p in enumerate(pairs):
        (s,), f = gpu_batch([p], api.PF_RGB_U8)
        assert s == scores[i] and np.array_equal(f[0], feats[i])
