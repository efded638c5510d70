"""Butteraugli's matrix-core strips (vship_amd/csrc/butter_strip.hip) hold
their precision: the distortion map against the FP64 oracle, on average over
its pixels.

The bounds come from the metric computed in FP32 on a CPU on these very inputs:
1.3e-6 of the mean map value with FP32 blurs, 2.1e-6 with blurs of operands
split into two fp16 parts, and at least 1.4e-4 with any of the products of a high and
a low part left out; the norms 7e-7, 2e-6 and 4e-5."""
import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests import butter_lib as bl
from tests.gpu_helpers import say
from tests.golden.make_golden import butter_inputs

pytestmark = pytest.mark.gpu

MAP_MEAN = 5e-6
NORM_RTOL = 1e-5


@pytest.mark.parametrize("w,h", [(64, 48), (130, 97), (257, 65), (256, 256)])
@pytest.mark.parametrize("seed", [31, 32])
def test_mean_map_error(w, h, seed):
    vship_amd.gpu_full_check(0)
    say(f"case mean map error {w}x{h}")
    ref, dist = butter_inputs(w, h, "f32", seed)
    want, wmap = bl.butteraugli(ref, dist, diffmap=True)
    dp = api.ButterDevicePairs([(ref, dist)], distmaps=True)
    try:
        with api.ButteraugliBatch(w, h, 1) as b:
            norms = b.compute(dp)[0]
        gmap = dp.distmap(0)
    finally:
        dp.free()
    mean = np.abs(gmap - wmap).mean() / wmap.mean()
    say(f"  map {mean:.1e} norms {np.abs(norms / want - 1).max():.1e}")
    assert mean <= MAP_MEAN
    assert np.all(np.abs(norms - want) <= NORM_RTOL * np.abs(want))
