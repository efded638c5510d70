// Map tiles of the FP64-moment class beside the matrix-core kernel: segments
// of fewer than kSmallSegmentMx pixels, whose FP32 rounding would not average
// out. What a tile computes is described at map_kernel (ssimu2_kernels.hip);
// here a workgroup of 256 threads takes one channel of a 16 x 16 tile, a
// thread per output pixel, so that the few pixels of these segments spread over
// many CUs: a 60 x 34 segment in two tiles of 32 x 48 with a workgroup per
// channel took 14.6 us, all of it the latency of one workgroup; ahead of the
// matrix-core tiles of the same launch these add 2 us.
#pragma once
#include <hip/hip_runtime.h>

#include "kernel_util.hpp"
#include "ssimu2_dev.hpp"

namespace vship {

struct SmallLds {
    static constexpr int kIn = kSmallTile + 16;  // input rows and columns
    float raw[2][kIn][kIn + 1];
    double h[4][kIn][kSmallTile + 1];  // row-pass results: a, b, (x1 - x2)^2, ab
    double red[4][6];
};

// Cumulative taps in FP64, for the renormalisation at image edges.
struct SmallCum {
    double v[18];
    constexpr SmallCum() : v() {
        for (int k = 0; k < 17; k++) v[k + 1] = v[k] + (double)tap(k);
    }
};
static __constant__ SmallCum kSmallCum{};

// Work item `item` (tile item / 3, channel item % 3) of the FP64 class of plane
// type ST. All 256 threads call it; L is free again after the last barrier.
template <typename ST>
__device__ __forceinline__ void map_small_tile(SmallLds& L, const PairDev* __restrict__ pairs,
                                               const int32_t* __restrict__ order_seg,
                                               const int32_t* __restrict__ order_start,
                                               const BatchHdr* __restrict__ hdr, const uint8_t* __restrict__ arena,
                                               double* __restrict__ partials, int item) {
    constexpr int grp = map_group(1, sizeof(ST) == 2), kIn = SmallLds::kIn;
    const int tid = threadIdx.x;
    int seg_lo = 0, t_begin = 0;
#pragma unroll
    for (int g = 0; g < grp; g++) {
        seg_lo += hdr->nseg[g];
        t_begin += hdr->tiles[g];
    }
    const int t = t_begin + item / 3, c = item % 3;
    int lo = seg_lo, hi = seg_lo + hdr->nseg[grp] - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (order_start[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    const int seg = order_seg[lo], s = seg % kScales;
    const PairDev& P = pairs[seg / kScales];
    const int W = P.sw[s], H = P.sh[s], pitch = P.pitch[s];
    const int ntx = (W + kSmallTile - 1) / kSmallTile, local = t - order_start[lo];
    const int y0 = local / ntx * kSmallTile, x0 = local % ntx * kSmallTile;
    const ST* p1 = reinterpret_cast<const ST*>(arena + P.arena_off + P.scale_off[s]) + c * P.plane_elems[s];
    const ST* p2 = reinterpret_cast<const ST*>(arena + P.arena_off + P.img_bytes + P.scale_off[s]) + c * P.plane_elems[s];
    // the 32 x 32 input samples of both images, at positions clamped into the
    // image, and the tile's centre value
    const double cc = (double)ldf(p1 + min(y0 + kSmallTile / 2, H - 1) * pitch + min(x0 + kSmallTile / 2, W - 1));
#pragma unroll
    for (int k = 0; k < 2 * kIn * kIn / 256; k++) {
        const int i = tid + 256 * k, col = i % kIn, row = i / kIn % kIn;
        const int o = min(max(y0 - 8 + row, 0), H - 1) * pitch + min(max(x0 - 8 + col, 0), W - 1);
        L.raw[i / (kIn * kIn)][row][col] = ldf((i < kIn * kIn ? p1 : p2) + o);
    }
    __syncthreads();
    // row pass: two neighbouring outputs of one of the 32 rows
    {
        const int r = tid >> 3, j0 = 2 * (tid & 7);
        const bool row_in = y0 - 8 + r >= 0 && y0 - 8 + r < H;
        double acc[4][2] = {};
#pragma unroll
        for (int k = 0; k < 18; k++) {
            const int x = x0 - 8 + j0 + k;
            const bool in = row_in && x >= 0 && x < W;
            const double u1 = (double)L.raw[0][r][j0 + k], u2 = (double)L.raw[1][r][j0 + k];
            const double a = in ? u1 - cc : 0.0, b = in ? u2 - cc : 0.0, d = in ? u1 - u2 : 0.0;
            const double v[4] = {a, b, d * d, a * b};
#pragma unroll
            for (int o = 0; o < 2; o++)
                if (k - o >= 0 && k - o <= 16)
#pragma unroll
                    for (int m = 0; m < 4; m++) acc[m][o] = fma((double)tap(k - o), v[m], acc[m][o]);
        }
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int o = 0; o < 2; o++) L.h[m][r][j0 + o] = acc[m][o];
    }
    __syncthreads();
    // column pass and the maps of this thread's pixel
    const int j = tid & 15, i = tid >> 4, x = x0 + j, y = y0 + i;
    double sum[6] = {};
    if (x < W && y < H) {
        double v[4] = {};
#pragma unroll
        for (int k = 0; k < 17; k++)
#pragma unroll
            for (int m = 0; m < 4; m++) v[m] = fma((double)tap(k), L.h[m][i + k][j], v[m]);
        const double iv = (1.0 / tap_total(kSmallCum.v, x, W)) * (1.0 / tap_total(kSmallCum.v, y, H));
        const double mu1 = v[0] * iv, mu2 = v[1] * iv, md = mu1 - mu2, md2 = md * md;
        const double vd = v[2] * iv - md2, num = fma(2.0, v[3] * iv - mu1 * mu2, 0.0009);
        const double d = fmax(fma(md2, num, vd) * (1.0 / (vd + num)), 0.0);
        const double a = (double)L.raw[0][i + 8][j + 8] - cc, b = (double)L.raw[1][i + 8][j + 8] - cc;
        const double fa = fabs(a - mu1) + 1.0, fb = fabs(b - mu2) + 1.0;
        const double ev = (fb - fa) * (1.0 / fa);
        const double art = fmax(ev, 0.0), det = fmax(-ev, 0.0);
        const double d2 = d * d, a2 = art * art, t2 = det * det;
        sum[0] = d;
        sum[1] = d2 * d2;
        sum[2] = art;
        sum[3] = a2 * a2;
        sum[4] = det;
        sum[5] = t2 * t2;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 6; k++) sum[k] += __shfl_xor(sum[k], off, 64);
    if ((tid & 63) == 0)
#pragma unroll
        for (int k = 0; k < 6; k++) L.red[tid >> 6][k] = sum[k];
    __syncthreads();
    if (tid < 6)
        partials[(int64_t)t * kFeat + c * 6 + tid] = ((L.red[0][tid] + L.red[1][tid]) + L.red[2][tid]) + L.red[3][tid];
}

}  // namespace vship
