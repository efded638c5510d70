"""Distortion maps of the per-frame Butteraugli handle on their way to host
memory (HostStager::download_rows, vship_amd/csrc/host_stage.hip): packed and
strided destinations of more than one staging chunk, rows longer than a chunk,
and several handles at once, whose planes and maps go by DMA where one handle's
go by a kernel. The maps equal the batched entry point's, written on the device."""
import ctypes
import threading

import numpy as np
import pytest

import vship_amd
from vship_amd import api
from tests.gpu_helpers import rgb_pair, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    vship_amd.gpu_full_check(0)
    yield


def device_map(ref, dist):
    h, w = ref[0].shape
    dp = api.ButterDevicePairs([(ref, dist)], distmaps=True)
    try:
        with api.ButteraugliBatch(w, h, 1) as b:
            b.compute(dp)
        return dp.distmap(0)
    finally:
        dp.free()


def host_map(handle, ref, dist, pad=0):
    """The map in rows of w + pad floats, the pad untouched."""
    h, w = ref[0].shape
    out = np.full((h, w + pad), -1.0, np.float32)
    score = api.ButterScore()
    rc = api.lib().Vship_ComputeButteraugliFloatv2(
        handle._h, ctypes.byref(score), out.ctypes.data, out.strides[0], api._plane_ptrs(ref), api._plane_ptrs(dist),
        ref[0].strides[0], dist[0].strides[0])
    assert rc == 0
    assert np.all(out[:, w:] == -1.0)
    return out[:, :w]


# one chunk of the ring is 2 MiB: 3.7 MB maps whose chunks start at every
# alignment of four bytes, and rows of 2.1 MB
@pytest.mark.parametrize("w,h,pad", [(1279, 719, 0), (1279, 719, 16), (1280, 720, 0), (530000, 3, 0), (530000, 3, 5)])
def test_map_to_host(w, h, pad):
    say(f"case map download {w}x{h} pad {pad}")
    if w > 4096:
        rng = np.random.default_rng(1)
        ref = [rng.random((h, w), np.float32) for _ in range(3)]
        dist = [np.clip(p + np.float32(0.02), 0, 1) for p in ref]
    else:
        ref, dist = rgb_pair(w, h, api.PF_RGB_F32, 7)
    want = device_map(ref, dist)
    with api.ButteraugliHandler(w, h) as handle:
        for _ in range(2):
            assert np.array_equal(host_map(handle, ref, dist, pad), want)


def test_handles_on_several_threads():
    say("case maps of four handles on four threads")
    w, h, n = 1279, 719, 4
    pairs = [rgb_pair(w, h, api.PF_RGB_F32, 10 + i) for i in range(n)]
    want = [device_map(*p) for p in pairs]
    handles = [api.ButteraugliHandler(w, h) for _ in range(n)]
    bad = []

    def work(i):
        for k in range(6):
            if not np.array_equal(host_map(handles[i], *pairs[i], pad=3 * (k & 1)), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for hd in handles:
        hd.close()
    assert not bad
