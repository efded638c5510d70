"""Workloads that stand for the use of this library, and what 64-bit
arithmetic gives for them.

A case scores frame pairs with one of the two metrics through one of the
public entry points of `vship_amd.api`:

  entry "device"  frames already in GPU memory (a GPU decoder, a renderer, a
                  tensor), one `SSIMU2Batch.compute` / `ButteraugliBatch.compute`
  entry "host"    frames in ordinary host memory, one per-frame call of the
                  drop-in handle (`SSIMU2Handler`, `ButteraugliHandler`)

The frames are synthetic: a picture of several octaves of noise with hard
edges that moves two pixels per frame, and a distorted copy of it, quantised
in 8 x 8 blocks, half of the blocks blurred. Scores come back as one float32
array per call, as a program keeps one float per frame (the planes they are
summed from are FP32); distortion maps are the float32 device tensors or host
arrays that the call fills; the drop-in Butteraugli score is three ints.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from vship_amd import api

DEVICE = "cuda"

# pixel format name -> (code, bits, log2 horizontal / vertical chroma subsampling; None: RGB)
FORMATS = {
    "rgb8": (api.PF_RGB_U8, 8, None),
    "rgb16": (api.PF_RGB_U16, 16, None),
    "rgbf16": (api.PF_RGB_F16, 0, None),
    "rgbf32": (api.PF_RGB_F32, 0, None),
    "yuv420p8": (api.PF_YUV420_U8, 8, (1, 1)),
    "yuv420p10": (api.PF_YUV420_U16, 10, (1, 1)),
    "yuv422p10": (api.PF_YUV422_U16, 10, (1, 0)),
    "yuv444p8": (api.PF_YUV444_U8, 8, (0, 0)),
}
MATRICES = {"bt709": (api.MATRIX_BT709, 0.2126, 0.0722), "bt2020": (api.MATRIX_BT2020NCL, 0.2627, 0.0593)}
# frame sizes of an uneven batch: the usual ladder of a stream, and cropped, odd ones
LADDER = [(640, 360), (1280, 720), (1920, 1080), (854, 479), (1919, 801), (2560, 1440), (426, 240), (3840, 2160)]


def _case(name, metric, entry, width, height, pairs, fmt, matrix="bt709", fp16=False, maps=False, mixed=False,
          qnorm=2):
    c = dict(metric=metric, entry=entry, width=width, height=height, pairs=pairs, fmt=fmt, matrix=matrix, fp16=fp16,
             maps=maps, mixed=mixed, qnorm=qnorm)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a thumbnail or a patch in an image-quality loop: the smallest call, all latency
        _case("ssimu2-256-rgb8", "ssimu2", "device", 256, 256, 1, "rgb8"),
        # an image tool on the drop-in interface: one picture pair of odd size from host memory
        _case("ssimu2-odd-host-rgb16", "ssimu2", "host", 1279, 719, 1, "rgb16"),
        # a video filter that scores frame by frame: one full-HD pair per call
        _case("ssimu2-1080p-single", "ssimu2", "device", 1920, 1080, 1, "yuv420p8"),
        # scoring an encode: the benchmark's batch of full-HD 4:2:0 pairs
        _case("ssimu2-1080p-batch240", "ssimu2", "device", 1920, 1080, 240, "yuv420p8"),
        # HDR masters: 4K 10-bit BT.2020, half-precision storage of the fine planes
        _case("ssimu2-4k10-fp16-batch24", "ssimu2", "device", 3840, 2160, 24, "yuv420p10", "bt2020", fp16=True),
        # the rungs of a bitrate ladder, and odd crops, in one call
        _case("ssimu2-mixed-batch32", "ssimu2", "device", 3840, 2160, 32, "yuv420p8", mixed=True),
        # intermediate (mezzanine) video: 4:2:2 10-bit, a short run of frames
        _case("ssimu2-1080p-422-batch8", "ssimu2", "device", 1920, 1080, 8, "yuv422p10"),
        # a thumbnail or a patch with Butteraugli
        _case("butter-256-rgb16", "butter", "device", 256, 256, 1, "rgb16"),
        # an image tool on the drop-in interface with the distortion map, odd size, from host memory
        _case("butter-odd-host-rgb16-map", "butter", "host", 1279, 719, 1, "rgb16", maps=True),
        # a filter that shows the distortion map of a full-HD float RGB pair
        _case("butter-1080p-single-map", "butter", "device", 1920, 1080, 1, "rgbf32", maps=True),
        # scoring an encode: the benchmark's batch of full-HD 4:2:0 pairs
        _case("butter-1080p-batch16", "butter", "device", 1920, 1080, 16, "yuv420p8"),
        # HDR masters: a few 4K 10-bit BT.2020 pairs, 3-norm as the Q-norm
        _case("butter-4k10-batch4", "butter", "device", 3840, 2160, 4, "yuv420p10", "bt2020", qnorm=3),
    ]


def draw(rng):
    """One more case of the same ranges: frames of 64 x 64 to 4K, one pair to a batch, every listed format."""
    metric = rng.choice(["ssimu2", "butter"])
    width = int(round(math.exp(rng.uniform(math.log(64), math.log(3840)))))
    height = max(64, min(2160, int(round(width * rng.uniform(0.5, 0.8)))))
    entry = rng.choice(["device", "device", "device", "host"])
    if entry == "host":
        return _case(None, metric, "host", width, height, 1, rng.choice(["rgb16", "rgbf32"]),
                     maps=metric == "butter", qnorm=rng.choice([2, 3]))
    # batches of at most 240 (16 for Butteraugli) full-HD pairs' pixels
    most = (240 if metric == "ssimu2" else 16) * 1920 * 1080 // (width * height)
    pairs = int(round(math.exp(rng.uniform(0.0, math.log(max(1, min(most, 240 if metric == "ssimu2" else 16)))))))
    fmt = rng.choice(sorted(FORMATS))
    matrix = "bt2020" if fmt == "yuv420p10" else "bt709"
    if metric == "butter":
        return _case(None, metric, entry, width, height, pairs, fmt, matrix, maps=rng.random() < 0.4,
                     qnorm=rng.choice([2, 3]))
    return _case(None, metric, entry, width, height, pairs, fmt, matrix, fp16=width > 1920 and rng.random() < 0.5)


def _sizes(case):
    if not case["mixed"]:
        return [(case["width"], case["height"])] * case["pairs"]
    return [LADDER[i % len(LADDER)] for i in range(case["pairs"])]


# ---------------------------------------------------------------------------
# frames
# ---------------------------------------------------------------------------
def _picture(w, h, gen):
    """A still [3, h, w] in [0, 1]: octaves of noise of falling amplitude, some hard-edged boxes."""
    out = torch.zeros(3, h, w, device=DEVICE)
    for cell, amp in ((96, 1.1), (24, 0.5), (6, 0.22), (1, 0.05)):
        n = torch.randn(1, 3, h // cell + 3, w // cell + 3, generator=gen, device=DEVICE)
        if cell > 1:
            n = F.interpolate(n, scale_factor=cell, mode="bilinear", align_corners=False)
        grey = n.mean(1, keepdim=True) * 1.5
        out += amp * (0.7 * grey + 0.3 * n)[0, :, :h, :w]
    box = torch.rand(12, 4, generator=gen, device=DEVICE).tolist()
    level = torch.randn(12, 3, 1, 1, generator=gen, device=DEVICE)
    for (x, y, bw, bh), lv in zip(box, level):
        x0, y0 = int(x * w), int(y * h)
        out[:, y0:y0 + 1 + int(bh * h / 4), x0:x0 + 1 + int(bw * w / 4)] += 0.8 * lv
    return torch.sigmoid(out)


def _distort(x, gen):
    """The picture after block coding: detail of 8 x 8 blocks quantised, half of the blocks blurred."""
    h, w = x.shape[1:]
    p = F.pad(x[None], (0, -w % 8, 0, -h % 8), mode="replicate")
    mean = F.interpolate(F.avg_pool2d(p, 8), scale_factor=8)
    by, bx = p.shape[2] // 8, p.shape[3] // 8
    r = torch.rand(2, 1, 1, by, bx, generator=gen, device=DEVICE)
    step = F.interpolate(0.02 + 0.06 * r[0], scale_factor=8)
    coded = mean + step * torch.round((p - mean) / step)
    soft = F.avg_pool2d(F.pad(coded, (1, 1, 1, 1), mode="replicate"), 3, stride=1)
    pick = F.interpolate((r[1] < 0.5).float(), scale_factor=8)
    return (coded + pick * (soft - coded))[0, :, :h, :w]


def _encode(x, case):
    """The three planes of the case's pixel format of a [3, h, w] picture in [0, 1]."""
    fmt = case["fmt"]
    _, bits, sub = FORMATS[fmt]
    x = x.clamp(0, 1)
    if fmt == "rgbf32":
        return [p.contiguous() for p in x]
    if fmt == "rgbf16":
        return [p.contiguous() for p in x.half()]
    if sub is None:
        q = torch.round(x * ((1 << bits) - 1)).to(torch.int32)
        return [p.contiguous() for p in q.to(torch.uint8 if bits == 8 else torch.uint16)]
    _, kr, kb = MATRICES[case["matrix"]]
    luma = kr * x[0] + (1 - kr - kb) * x[1] + kb * x[2]
    planes = [luma, (x[2] - luma) / (2 - 2 * kb), (x[0] - luma) / (2 - 2 * kr)]
    s, out = 1 << (bits - 8), []
    for i, p in enumerate(planes):
        if i and (sub[0] or sub[1]):
            fx, fy = 1 << sub[0], 1 << sub[1]
            h, w = p.shape
            p = F.avg_pool2d(F.pad(p[None, None], (0, -w % fx, 0, -h % fy), mode="replicate"), (fy, fx))[0, 0]
        q = p * (224 * s) + 128 * s if i else p * (219 * s) + 16 * s
        q = torch.round(q).clamp(0, (1 << bits) - 1).to(torch.int32)
        out.append(q.to(torch.uint8 if bits == 8 else torch.uint16).contiguous())
    return out


def _frames(case, seed):
    """The case's pairs: (reference planes, distorted planes), tensors on the GPU."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    stills, out = {}, []
    for i, (w, h) in enumerate(_sizes(case)):
        if (w, h) not in stills:
            stills[w, h] = _picture(w + 64, h, gen)
        at = 2 * i % 64
        ref = stills[w, h][:, :, at:at + w]
        out.append((_encode(ref, case), _encode(_distort(ref, gen), case)))
    return out


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
class State:
    """What a program keeps between calls: its frames, their descriptors and the handle."""

    handle = None

    def __del__(self):
        if self.handle is not None:
            self.handle.close()


class DevicePairs:
    """Butteraugli descriptors of frames in tensors, as `ButteraugliBatch.compute` takes them."""


def _point(desc, ref, dist):
    for k in range(3):
        desc.ref[k], desc.dist[k] = ref[k].data_ptr(), dist[k].data_ptr()
        desc.ref_stride[k] = ref[k].stride(0) * ref[k].element_size()
        desc.dist_stride[k] = dist[k].stride(0) * dist[k].element_size()


def prepare(case, seed):
    s = State()
    s.case = case
    s.frames = _frames(case, seed)
    s.maps = None
    code, bits, sub = FORMATS[case["fmt"]]
    n, w, h = case["pairs"], case["width"], case["height"]
    if case["entry"] == "host":
        s.frames = [([p.cpu().numpy() for p in r], [p.cpu().numpy() for p in d]) for r, d in s.frames]
        s.handle = api.SSIMU2Handler(w, h) if case["metric"] == "ssimu2" else api.ButteraugliHandler(w, h, case["qnorm"])
        return s
    matrix = MATRICES[case["matrix"]][0]
    if case["metric"] == "ssimu2":
        s.descs = (api.Pair * n)()
        for d, (ref, dist) in zip(s.descs, s.frames):
            _point(d, ref, dist)
            d.height, d.width = ref[0].shape
            d.format, d.bits, d.matrix, d.chroma_location = code, bits, matrix, api.CHROMA_LEFT
        s.handle = api.SSIMU2Batch(n, w, h, fp16=case["fp16"])
    else:
        s.descs = (api.ButterPair * n)()
        if case["maps"]:
            s.maps = [torch.zeros(h, w, device=DEVICE) for _ in range(n)]
        for i, (d, (ref, dist)) in enumerate(zip(s.descs, s.frames)):
            _point(d, ref, dist)
            d.bits, d.matrix, d.chroma_location = bits, matrix, api.CHROMA_LEFT
            if s.maps:
                d.distmap, d.distmap_stride = s.maps[i].data_ptr(), w * 4
        s.pairs = DevicePairs()
        s.pairs.format, s.pairs.descs, s.pairs.n = code, s.descs, n
        s.handle = api.ButteraugliBatch(w, h, n, qnorm=case["qnorm"])
    torch.cuda.synchronize()  # the library works on streams of its own
    return s


def run(state):
    c, h = state.case, state.handle
    if c["entry"] == "host":
        ref, dist = state.frames[0]
        if c["metric"] == "ssimu2":
            return (h.compute_float if c["fmt"] == "rgbf32" else h.compute_uint16)(ref, dist)
        return (h.compute_float if c["fmt"] == "rgbf32" else h.compute_uint16)(ref, dist, distmap=c["maps"])
    if c["metric"] == "ssimu2":
        return h.compute(state.descs).astype(np.float32)
    norms = h.compute(state.pairs).astype(np.float32)
    return {"norms": norms, "maps": state.maps} if state.maps else norms


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every input sample once, every score and map once. Flops: the
    metric's own sums, counted per pixel of each scale of a pair."""
    _, bits, sub = FORMATS[case["fmt"]]
    size = 4 if case["fmt"] == "rgbf32" else 1 if bits == 8 else 2
    chroma = 1.0 if sub is None else 1.0 / (1 << (sub[0] + sub[1]))
    nbytes = flops = 0.0
    for w, h in _sizes(case):
        nbytes += 2 * size * w * h * (1 + 2 * chroma)
        if case["metric"] == "ssimu2":
            # three channels: four blurred moments (two passes of 17 taps), about 40 for the maps and their sums
            nbytes += 8
            flops += w * h * 4 / 3 * 3 * (4 * 2 * 17 * 2 + 40)
        else:
            # blurs: 17 taps on 6 planes, 43 on 6, 19 on 6, 17 on 4, 17 on 2, two passes each;
            # Malta lines 2 x (128 + 32) + 4 x (80 + 32); about 300 for the points
            nbytes += 24 + (4 * w * h if case["maps"] else 0)
            flops += w * h * 5 / 4 * (4 * (6 * 17 + 6 * 43 + 6 * 19 + 4 * 17 + 2 * 17) + 768 + 300)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# 64-bit values: planes are [..., h, w] float64 tensors
# ---------------------------------------------------------------------------
def _shifted(x, k, dim):
    """y[i] = x[i + k] along dim, 0 where i + k lies outside."""
    n = x.shape[dim]
    y = torch.zeros_like(x)
    if abs(k) < n:
        y.narrow(dim, max(0, -k), n - abs(k)).copy_(x.narrow(dim, max(0, k), n - abs(k)))
    return y


def _blur(x, sigma, radius):
    """Gaussian over the samples inside the image, each axis divided by the taps that lie inside."""
    g = [math.exp(-k * k / (2 * sigma * sigma)) for k in range(-radius, radius + 1)]
    for dim in (-1, -2):
        n = x.shape[dim]
        acc, tot = torch.zeros_like(x), torch.zeros(n, dtype=torch.float64, device=x.device)
        for k in range(-radius, radius + 1):
            if abs(k) >= n:
                continue
            lo, src, m = max(0, -k), max(0, k), n - abs(k)
            acc.narrow(dim, lo, m).add_(x.narrow(dim, src, m), alpha=g[k + radius])
            tot[lo:lo + m] += g[k + radius]
        x = acc / (tot if dim == -1 else tot[:, None])
    return x


def _halve(x):
    """2 x 2 means, the last row and column repeated where the size is odd."""
    h, w = x.shape[-2:]
    x = F.pad(x, (0, w % 2, 0, h % 2), mode="replicate")
    return 0.25 * (x[..., ::2, ::2] + x[..., 1::2, ::2] + x[..., ::2, 1::2] + x[..., 1::2, 1::2])


def _upsample(p, n, shift, centred, dim):
    """Catmull-Rom samples at the n luma positions of an axis subsampled by 2^shift, edge samples repeated."""
    if not shift:
        return p
    f = 1 << shift
    x = torch.arange(n, dtype=torch.float64, device=p.device)
    u = (x - (f - 1) / 2) / f if centred else x / f
    base = u.floor()
    t = u - base
    ws = [0.5 * t * ((2 - t) * t - 1), 0.5 * ((3 * t - 5) * t * t + 2), 0.5 * t * ((4 - 3 * t) * t + 1),
          0.5 * t * t * (t - 1)]
    out = 0
    for k, wk in enumerate(ws):
        at = (base.long() + k - 1).clamp(0, p.shape[dim] - 1)
        out = out + p.index_select(dim, at) * (wk if dim == -1 else wk[:, None])
    return out


def _linear(planes, case):
    """Linear RGB [3, h, w] of a frame's planes."""
    fmt = case["fmt"]
    _, bits, sub = FORMATS[fmt]
    x = [(p if p.is_floating_point() else p.to(torch.int32)).double() for p in planes]
    if sub is None:
        rgb = torch.stack(x)
        if bits:
            rgb = rgb / ((1 << bits) - 1)
    else:
        _, kr, kb = MATRICES[case["matrix"]]
        s = 1 << (bits - 8)
        h, w = x[0].shape
        y = (x[0] - 16 * s) / (219 * s)
        cb, cr = ((_upsample(_upsample(p, w, sub[0], False, -1), h, sub[1], True, -2) - 128 * s) / (224 * s)
                  for p in x[1:])
        r, b = y + 2 * (1 - kr) * cr, y + 2 * (1 - kb) * cb
        rgb = torch.stack([r, (y - kr * r - kb * b) / (1 - kr - kb), b])
    return torch.sign(rgb) * rgb.abs() ** 2.4


# The published SSIMULACRA2 weights: channel X, Y, B; per scale the 1-norms of
# the similarity, artifact and detail-loss maps, then their 4-norms.
_SSIMU2_WEIGHTS = [
    0.0, 0.0007376606707406586, 0.0, 0.0, 0.0007793481682867309, 0.0,
    0.0, 0.0004371155730107379, 0.0, 1.1041726426657346, 0.00066284834129271, 0.00015231632783718752,
    0.0, 0.0016406437456599754, 0.0, 1.8422455520539298, 11.441172603757666, 0.0,
    0.0007989109436015163, 0.000176816438078653, 0.0, 1.8787594979546387, 10.94906990605142, 0.0,
    0.0007289346991508072, 0.9677937080626833, 0.0, 0.00014003424285435884, 0.9981766977854967, 0.00031949755934435053,
    0.0004550992113792063, 0.0, 0.0, 0.0013648766163243398, 0.0, 0.0,
    0.0, 0.0, 0.0, 7.466890328078848, 0.0, 17.445833984131262,
    0.0006235601634041466, 0.0, 0.0, 6.683678146179332, 0.00037724407979611296, 1.027889937768264,
    225.20515300849274, 0.0, 0.0, 19.213238186143016, 0.0011401524586618361, 0.001237755635509985,
    176.39317598450694, 0.0, 0.0, 24.43300999870476, 0.28520802612117757, 0.0004485436923833408,
    0.0, 0.0, 0.0, 34.77906344483772, 44.835625328877896, 0.0,
    0.0, 0.0, 0.0, 0.0, 0.0, 0.0,
    0.0, 0.0008680556573291698, 0.0, 0.0, 0.0, 0.0,
    0.0, 0.0005313191874358747, 0.0, 0.00016533814161379112, 0.0, 0.0,
    0.0, 0.0, 0.0, 0.0004179171803251336, 0.0017290828234722833, 0.0,
    0.0020827005846636437, 0.0, 0.0, 8.826982764996862, 23.19243343998926, 0.0,
    95.1080498811086, 0.9863978034400682, 0.9834382792465353, 0.0012286405048278493, 171.2667255897307, 0.9807858872435379,
    0.0, 0.0, 0.0, 0.0005130064588990679, 0.0, 0.00010854057858411537,
]


def _positive_xyb(rgb):
    r, g, b = rgb
    bias, root = 0.0037930734, -0.1559542025327239
    lms = [0.30 * r + 0.622 * g + 0.078 * b, 0.23 * r + 0.692 * g + 0.078 * b,
           0.24342269 * r + 0.20476745 * g + 0.55180986 * b]
    l, m, s = ((v + bias).clamp(min=0) ** (1 / 3) + root for v in lms)
    x, y = 0.5 * (l - m), 0.5 * (l + m)
    return torch.stack([14 * x + 0.42, y + 0.01, (s - y) + 0.55])


def _ssimu2(a, b):
    feats = torch.zeros(3, 6, 2, 3, dtype=torch.float64, device=a.device)
    for s in range(6):
        if s:
            a, b = _halve(a), _halve(b)
        x, y = _positive_xyb(a), _positive_xyb(b)
        mx, my, xx, yy, xy = _blur(torch.stack([x, y, x * x, y * y, x * y]), 1.5, 8)
        d = 1 - (1 - (mx - my) ** 2) * (2 * (xy - mx * my) + 0.0009) / ((xx - mx * mx) + (yy - my * my) + 0.0009)
        e = ((y - my).abs() + 1) / ((x - mx).abs() + 1) - 1
        for m, v in enumerate((d.clamp(min=0), e.clamp(min=0), (-e).clamp(min=0))):
            feats[:, s, 0, m] = v.mean((-1, -2))
            feats[:, s, 1, m] = (v ** 4).mean((-1, -2)) ** 0.25
    q = 0.9562382616834844 * float(np.dot(feats.flatten().cpu().numpy(), np.array(_SSIMU2_WEIGHTS)))
    q = 6.248496625763138e-5 * q ** 3 - 0.020884521182843837 * q * q + 2.326765642916932 * q
    return 100 - 10 * q ** 0.6276336467831387 if q > 0 else 100.0


def _lines(*halves):
    """Line filters from the taps on one side of the centre (dx, dy): point-symmetric unless a pair of lists is given."""
    out = []
    for h in halves:
        one, other = h if isinstance(h, tuple) else (h, [(-x, -y) for x, y in h])
        out.append(one + [(0, 0)] + other)
    return out


def _all_lines(horizontal, diagonal, steep, slanted, bent):
    """The sixteen directions of a Malta filter from one line of each kind, by reflection and transposition."""
    def flip(h, fx=1, fy=1, swap=False):
        def one(v):
            v = [(y, x) if swap else (x, y) for x, y in v]
            return [(fx * x, fy * y) for x, y in v]
        return tuple(one(v) for v in h) if isinstance(h, tuple) else one(h)
    return _lines(horizontal, flip(horizontal, swap=True), diagonal, flip(diagonal, fx=-1),
                  steep, flip(steep, fx=-1), flip(steep, swap=True), flip(steep, fx=-1, swap=True),
                  slanted, flip(slanted, fx=-1), flip(slanted, swap=True), flip(slanted, fx=-1, swap=True),
                  bent, flip(bent, fy=-1), flip(bent, swap=True), flip(bent, fx=-1, swap=True))


_MALTA_FINE = _all_lines([(-4, 0), (-3, 0), (-2, 0), (-1, 0)], [(-3, -3), (-2, -2), (-1, -1)],
                         [(1, -4), (1, -3), (1, -2), (0, -1)], [(-2, -3), (-1, -2), (-1, -1)],
                         ([(-4, -2), (-3, -2), (-2, -1), (-1, -1)], [(1, 0), (2, 1), (3, 1)]))
_MALTA_COARSE = _all_lines([(-4, 0), (-2, 0)], [(-3, -3), (-2, -2)], [(1, -4), (1, -2)], [(-2, -3), (-1, -2)],
                           [(-4, -2), (-2, -1)])


def _outside(a, b, low, high):
    """How far b lies outside [low |a|, high |a|] on a's side."""
    m = torch.where(a < 0, -b, b)
    return (low * a.abs() - m).clamp(min=0) + (m - high * a.abs()).clamp(min=0)


def _malta(a, b, fine, gt, lt, norm):
    scale = (0.39905817637 if fine else 0.611612573796) / 8.5 * norm / (norm + 0.5 * a.abs() + 0.5 * b.abs())
    diff = a - b
    v = math.sqrt(0.5 * gt) * scale * diff
    v = v + torch.where(diff < 0, -1.0, 1.0) * math.sqrt(0.33 * lt) * scale * _outside(a, b, 0.55, 1.05)
    out = torch.zeros_like(v)
    for line in _MALTA_FINE if fine else _MALTA_COARSE:
        acc = torch.zeros_like(v)
        for dx, dy in line:
            acc += _shifted(_shifted(v, dx, -1), dy, -2)
        out += acc * acc
    return out


def _asymmetric(a, b, gt, lt):
    return 0.8 * (gt * (a - b) ** 2 + lt * _outside(a, b, 0.4, 1.0) ** 2)


def _shrink(x, w):
    return torch.where(x > w, x - w, torch.where(x < -w, x + w, torch.zeros_like(x)))


def _grow(x, w):
    return torch.where(x > w, x + w, torch.where(x < -w, x - w, 2 * x))


def _soft_clamp(x, top):
    c = x.clamp(-top, top)
    return c + 0.688059627878 * (x - c)


_OPSIN = [(0.29956550340058319, 0.63373087833825936, 0.077705617820981968, 1.7557483643287353),
          (0.22158691104574774, 0.69391388044116142, 0.0987313588422, 1.7557483643287353),
          (0.02, 0.02, 0.20480129041026129, 12.226454707163354)]


def _bands(lin):
    """Low, middle (X, Y, B), high and ultra-high (X, Y) bands of a linear RGB picture at 203 nits."""
    sharp, soft = 203.0 * lin, 203.0 * _blur(lin, 1.2, 8)
    cones = []
    for r, g, b, k in _OPSIN:
        v = (r * soft[0] + g * soft[1] + b * soft[2] + k).clamp(min=k)
        gain = ((19.245013259874995 * torch.log(v + 9.9710635769299145) - 23.16046239805755) / v).clamp(min=1e-4)
        cones.append(((r * sharp[0] + g * sharp[1] + b * sharp[2] + k) * gain).clamp(min=k))
    xyb = torch.stack([cones[0] - cones[1], cones[0] + cones[1], cones[2]])
    low = _blur(xyb, 7.15593339443, 21)
    rest = xyb - low
    mid = _blur(rest, 3.22489901262, 9)
    high = (rest - mid)[:2]
    mid = torch.stack([_shrink(mid[0], 0.29), _grow(mid[1], 0.1), mid[2]])
    keep = 0.653020556257
    high = torch.stack([high[0] * (keep + 46.0 * (1 - keep) / (46.0 + high[1] ** 2)), high[1]])
    smooth = _blur(high, 1.56416327805, 8)
    hy = _soft_clamp(smooth[1], 28.4691806922)
    uhf = torch.stack([_shrink(high[0] - smooth[0], 0.04),
                       2.69313763794 * _soft_clamp(high[1] - hy, 5.19175294647)])
    hf = torch.stack([_shrink(smooth[0], 1.5), _grow(2.155 * hy, 0.132)])
    low = torch.stack([33.832837186260 * low[0], 14.458268100570 * low[1],
                       49.87984651440 * (low[2] - 0.362267051518 * low[1])])
    return low, mid, hf, uhf


def _erode(x):
    """0.45, 0.3 and 0.25 of the three smallest values among a pixel, twice it, and its neighbours three pixels away."""
    cand = [x, 2 * x, 2 * x]
    h, w = x.shape
    inside = torch.ones_like(x)
    for dx in (-3, 0, 3):
        for dy in (-3, 0, 3):
            if dx or dy:
                v = _shifted(_shifted(x, dx, -1), dy, -2)
                ok = _shifted(_shifted(inside, dx, -1), dy, -2) > 0
                cand.append(torch.where(ok, v, torch.full_like(x, math.inf)))
    m = torch.stack(cand).topk(3, dim=0, largest=False).values
    return 0.45 * m[0] + 0.3 * m[1] + 0.25 * m[2]


def _butter_map(a, b):
    (la, ma, ha, ua), (lb, mb, hb, ub) = _bands(a), _bands(b)
    s = 0.8
    r = math.sqrt(s)
    ac = (_malta(ua[1], ub[1], True, 1.10039032555 * s, 1.10039032555 / s, 71.7800275169)
          + _malta(ua[0], ub[0], True, 173.5 * s, 173.5 / s, 5.0)
          + _malta(ha[1], hb[1], False, 18.7237414387 * r, 18.7237414387 / r, 4498534.45232)
          + _malta(ha[0], hb[0], False, 6923.99476109 * r, 6923.99476109 / r, 8051.15833247)
          + _malta(ma[1], mb[1], False, 37.0819870399, 37.0819870399, 130262059.556)
          + _malta(ma[0], mb[0], False, 8246.75321353, 8246.75321353, 1009002.70582)
          + _asymmetric(ha[0], hb[0], 400.0 * s, 400.0 / s)
          + _asymmetric(ha[1], hb[1], 1.50815703118 * s, 1.50815703118 / s))
    dc = torch.zeros_like(ac)
    for c in range(3):
        ac += (2150.0, 10.6195433239, 16.2176043152)[c] * (ma[c] - mb[c]) ** 2
        dc += (29.2353797994, 0.844626970982, 0.703646627719)[c] * (la[c] - lb[c]) ** 2
    blurred = []
    for h, u in ((ha, ua), (hb, ub)):
        amp = torch.sqrt((2.5 * (u[0] + h[0])) ** 2 + (0.4 * (u[1] + h[1])) ** 2)
        bias = 6.19424080439 * 12.61050594197
        blurred.append(_blur(torch.sqrt(6.19424080439 * amp + bias) - math.sqrt(bias), 2.7, 8))
    ac += 10.0 * (blurred[0] - blurred[1]) ** 2
    mask, norm = _erode(blurred[0]), 1.0 / (0.79079917404 * 17.83)
    way = ((1 + 2.5485944793 / (0.451936922203 * mask + 0.829591754942)) * norm) ** 2
    wdc = ((1 + 0.505054525019 / (3.87449418804 * mask + 0.20025578522)) * norm) ** 2
    return torch.sqrt(way * ac + wdc * dc)


def _butter(a, b, qnorm):
    full, half = _butter_map(a, b), _butter_map(_halve(a), _halve(b))
    h, w = full.shape
    v = 0.85 * full + 0.5 * half.repeat_interleave(2, 0).repeat_interleave(2, 1)[:h, :w]
    return v, [float((v ** q).mean() ** (1 / q)) for q in (qnorm, 3)] + [float(v.max())]


def exact(case, seed):
    if DEVICE == "cuda" and not torch.cuda.is_available():
        return None
    values, maps = [], []
    for ref, dist in _frames(case, seed):
        a, b = _linear(ref, case), _linear(dist, case)
        if case["metric"] == "ssimu2":
            values.append(_ssimu2(a, b))
        else:
            m, norms = _butter(a, b, case["qnorm"])
            values.append(norms)
            maps.append(m)
    if case["metric"] == "ssimu2":
        return values[0] if case["entry"] == "host" else np.array(values)
    if case["entry"] == "host":
        return ((None, None, None), maps[0]) if case["maps"] else (None, None, None)
    return {"norms": np.array(values), "maps": maps} if case["maps"] else np.array(values)
