"""The matrix-core map kernel's tiles of 64 x 128, two strips of 16 columns per
wave, at sizes that end on, before or after a strip, a wave's columns, a block of
rows, half a tile or a tile, and around the first interior tile: against the
FP64 oracle, and the same scores bit for bit however a launch shares the tiles
out (a wave per half of a tile's rows, a workgroup per channel, a workgroup per
tile)."""
import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests.gpu_helpers import gpu_batch, oracle_rgb, rgb_pair, say

pytestmark = pytest.mark.gpu

MFMA = 1
SCORE_ATOL = 1e-3  # the bar of every score against the oracle
SIZES = [(32, 128), (33, 129), (48, 127), (49, 144), (63, 145), (64, 64), (65, 65), (80, 192), (81, 193), (96, 257),
         (97, 256), (135, 263), (136, 264), (201, 280)]


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


@pytest.mark.parametrize("fmt", [api.PF_RGB_U8, api.PF_RGB_F32])
@pytest.mark.parametrize("w,h", SIZES)
def test_every_share_of_the_tiles(w, h, fmt):
    say(f"case shared windows {w}x{h} format {fmt}")
    ref, dist = rgb_pair(w, h, fmt, 3 * w + h)
    want, _ = oracle_rgb(ref, dist, fmt)
    for fp16 in (False, True):
        (got,), feats = gpu_batch([(ref, dist)], fmt, th=MFMA, fp16=fp16)
        # (FP16 planes of pictures this small move a score by more than the bar
        # before the kernel reads them: what they share is the tiles' arithmetic)
        assert fp16 or abs(got - want) <= SCORE_ATOL
        # a workgroup per tile
        (s,), f = gpu_batch([(ref, dist)], fmt, th=MFMA, fp16=fp16, persistent_grid=3)
        assert s == got and np.array_equal(f, feats)
    # enough tiles for a workgroup per channel with all rows to a wave
    (got,), feats = gpu_batch([(ref, dist)], fmt, th=MFMA)
    many = [(ref, dist)] * 1100
    scores, fs = gpu_batch(many, fmt, th=MFMA)
    assert np.all(scores == got) and np.all(fs == feats[0])
