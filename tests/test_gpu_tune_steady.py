"""The autotuner (vship_amd/csrc/tune.hip) times its candidates at the rate a
run of many batches has, not while the GPU comes out of idle."""
import time

import numpy as np
import pytest

import vship_amd
from vship_amd import api, synth
from tests.gpu_helpers import say

pytestmark = pytest.mark.gpu


def test_first_candidate_is_timed_at_its_steady_rate():
    """The first pass of a new engine takes 10 to 80 % more than later ones; one
    timed pass per candidate is enough where the warm-up has settled."""
    vship_amd.gpu_full_check(0)
    say("case tuner warm-up")
    clip = synth.video_clip(1920, 1080, 8, 1, seed=5)
    frame = clip.frame(0)
    clip.close()
    n = 48
    dp = api.DevicePairs([frame], api.PF_YUV420_U8, 8, 0)
    try:
        descs = (api.Pair * n)(*[dp.descs[0]] * n)
        tuned = api.autotune(descs, n, repeats=1)
        first = tuned["candidates"][0]
        assert first["persistent_grid"] == 0 and not first["use_graph"]
        with api.SSIMU2Batch(n, 1920, 1080, map_tile_height=first["map_tile_height"]) as b:
            t = []
            for _ in range(60):
                t0 = time.perf_counter()
                b.compute(descs)
                t.append((time.perf_counter() - t0) * 1e3)
        steady = float(np.median(t[20:]))
        say(f"  timed {first['ms']:.3f} ms, steady {steady:.3f}")
        assert first["ms"] <= 1.06 * steady
    finally:
        dp.free()
