// Map kernel on the gfx950 matrix cores, for the FP32-moment segments.
//
// Same result as map_kernel<TH, ST, float> (renormalised 17-tap Gaussian of
// the four moment planes a, b, (a - b)^2, ab of the samples centred per image
// on the tile-centre values (a = x1 - c1, b = x2 - c2), then the SSIM, artifact and
// detail-loss maps and their 1-/4-norm sums; src/ssimu2/gaussianblur.hpp:24-92,
// src/ssimu2/score.hpp:95-196), with both blur passes done as matrix products
// on the 16x16x32 MFMA instructions:
//
//   row pass    Hr(16 rows x 16 cols) = In(16 rows x 32 input cols) . G(32 x 16)
//   column pass Out(16 rows x 16 cols) = G'(16 x 32 input rows) . Hr(32 rows x 16 cols)
//
// where G[k][j] = g[k - j] (zero outside 0..16) is the band of taps; both
// passes use the same per-lane tap operand. The operands are split into
// 16-bit parts and the partial products accumulate in FP32, one of two ways:
//
//   SplitBf16x3 (planar float RGB input, whose values are unbounded): every
//     operand x is split exactly into three bf16 parts x = h + m + l
//     (truncation: h keeps the top 8 significant bits, m the next 8, l the
//     last 8); the six products above 2^-24 are accumulated (hh + hm + mh +
//     hl + mm + lh). FP32 accuracy, FP32 range.
//   SplitF16x2 (8- to 16-bit RGB and YUV input): operands are scaled by a
//     power of two (a, b and a - b: 2^2, so (a - b)^2 and ab: 2^4; taps:
//     2^14) and split into two fp16 parts h + l; the products hh + hl + lh
//     are accumulated, each exact (the lo x lo product, below the split's own
//     error, is dropped). A value whose low part is a normal fp16 number keeps
//     22 significant bits; a smaller one keeps an absolute error of at most
//     2^-25 at its scale (under 1e-8 in XYB units, far below the SSIM
//     constants 0.0009 these moments meet). The scales are the smallest
//     powers of two that need no multiply of their own (a and b come from
//     one FMA each, (a - b)^2 and ab are products of the scaled factors) and
//     they keep every value inside the fp16 range for any input of these
//     formats: their R'G'B' lies in [-0.97, 1.98] (limited-range YUV with
//     samples clamped to the declared depth), so XYB lies in [-11.7, 12.5] x
//     [-0.15, 1.58] x [-1.18, 2.28], |a|, |b| <= 24.2, |a - b| <= 48.4 and
//     |ab| <= 586, i.e. at most 37,500 at scale 2^4. The taps are the values
//     the fp16 pair represents exactly (within 2^-22 of the FP32 taps), and
//     the renormalisation sums use the same values. On the GPU the scores of
//     real frames stay within 3e-5 of the FP64 oracle, at about half the
//     splitting work of the exact split and two thirds of its matrix products.
//
// Tile: 64 columns x 128 rows of output pixels of one scale; each wave owns 32
// columns (144 input rows x 48 input columns) and needs nothing from the other
// waves until the tile sums. Its 48 input columns are three windows of 16, which
// two strips of 16 output columns share: the moments and splits of a window are
// made once and are half of each strip's operand, in place. The row-pass results
// stay in the lane whose column-pass operand they are half of, the other half
// being the block of rows before. Each output pixel's maps are formed in the
// registers the column pass leaves them in.
//
// What bounds it is power as much as vector issue: the chip holds about 2 GHz of
// its 2.4 in it, and less the more matrix products and memory traffic there are.
// With a wave per strip (each input column split twice: 370 issue slots of the
// vector unit per 16 x 16 outputs, 24 matrix products) the kernel took 7.53 ms for
// 240 1080p pairs; with shared windows and 325 slots 6.66 ms, 87 % of its cycles in
// vector issue and 26 % with the matrix cores busy. Forms with fewer slots and more
// products (28, 32) were no faster or slower, and 16 waves of this form per CU read
// the centre samples from beyond the L2, at a lower clock, for no gain until those
// came through LDS; twelve waves have the registers to load a window ahead. Memory
// is the other bound by now: for 240 1080p pairs the kernel reads 32.4 GB beyond
// the L2, where its planes hold 15.9 (a wave per strip read 18.4 GB), 4.8 TB/s.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "kernel_util.hpp"
#include "map_small.hpp"
#include "ssimu2_dev.hpp"
#include "ssimu2_kernels.hpp"

namespace vship {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// exact three-way bf16 split
// ---------------------------------------------------------------------------
__device__ __forceinline__ void split3(float x, float& h, float& m, float& l) {
    h = __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    const float r = x - h;
    m = __uint_as_float(__float_as_uint(r) & 0xffff0000u);
    l = r - m;
}

// Two bf16 values (the upper halves of two floats) in one word, the first in
// the low half.
__device__ __forceinline__ uint32_t pack2(float first, float second) {
    return __builtin_amdgcn_perm(__float_as_uint(second), __float_as_uint(first), 0x07060302u);
}

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

struct SplitBf16x3 {
    static constexpr int kParts = 3;
    static constexpr float kScaleAB = 1.f, kScaleDD = 1.f, kScaleQ = 1.f, kTapScale = 1.f;
    struct Op {
        u32x4 p[3];  // h, m, l
    };
    // N consecutive values
    template <int N>
    static __device__ __forceinline__ void split(const float* v, uint32_t (&w)[3][N / 2]) {
#pragma unroll
        for (int k = 0; k < N / 2; k++) {
            float h0, m0, l0, h1, m1, l1;
            split3(v[2 * k], h0, m0, l0);
            split3(v[2 * k + 1], h1, m1, l1);
            w[0][k] = pack2(h0, h1);
            w[1][k] = pack2(m0, m1);
            w[2][k] = pack2(l0, l1);
        }
    }
    // split of the four products x[e] y[e] (y = nullptr: of x[e])
    static __device__ __forceinline__ void split_prod4(const float* x, const float* y, uint32_t (&w)[3][2]) {
        float p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) p[k] = y ? x[k] * y[k] : x[k];
        split<4>(p, w);
    }
    // split of x * s (row-pass results, re-split at the data scale)
    template <int N>
    static __device__ __forceinline__ void split_scaled(const float* v, float s, uint32_t (&w)[3][N / 2]) {
        float x[N];
#pragma unroll
        for (int k = 0; k < N; k++) x[k] = v[k] * s;
        split<N>(x, w);
    }
    // c + a.b from the six partial products above 2^-24, smallest first
    static __device__ __forceinline__ f32x4 mma(const Op& a, const Op& b, f32x4 c) {
        c = mfma_bf16(a.p[2], b.p[0], c);
        c = mfma_bf16(a.p[1], b.p[1], c);
        c = mfma_bf16(a.p[0], b.p[2], c);
        c = mfma_bf16(a.p[1], b.p[0], c);
        c = mfma_bf16(a.p[0], b.p[1], c);
        c = mfma_bf16(a.p[0], b.p[0], c);
        return c;
    }
    static __device__ __forceinline__ float tap_value(int k) { return tap(k); }
};

// ---------------------------------------------------------------------------
// scaled two-way fp16 split
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

struct SplitF16x2 {
    static constexpr int kParts = 2;
    static constexpr float kScaleAB = 4.f;  // a, b: 2^2
    static constexpr float kScaleDD = 4.f;  // (a - b)^2 as (4 (a - b))^2: 2^4
    static constexpr float kScaleQ = 1.f;   // ab from the scaled a, b: 2^4
    static constexpr float kTapScale = 16384.f;      // taps: 2^14
    struct Op {
        u32x4 p[2];  // h, l
    };
    template <int N>
    static __device__ __forceinline__ void split(const float* v, uint32_t (&w)[2][N / 2]) {
#pragma unroll
        for (int k = 0; k < N / 2; k++) {
            const f32x2 x = {v[2 * k], v[2 * k + 1]};
            const f16x2 h = __builtin_convertvector(x, f16x2);
            const f32x2 r = x - __builtin_convertvector(h, f32x2);
            const f16x2 l = __builtin_convertvector(r, f16x2);
            w[0][k] = __builtin_bit_cast(uint32_t, h);
            w[1][k] = __builtin_bit_cast(uint32_t, l);
        }
    }
    // split of the four products x[e] y[e] (y = nullptr: of x[e]): h = fp16(x y)
    // by the compiler; the low parts
    // l = fp16(x y - h), each one v_fma_mixlo/mixhi_f16 that forms x y - h
    // exactly and rounds once, written by inline assembly (the compiler
    // splits them into a multiply-subtract and a conversion). The block ends
    // with s_nop 1: the compiler counts no VALU wait states for inline
    // assembly, and a matrix-core instruction reading a register a VALU
    // instruction wrote needs two.
    static __device__ __forceinline__ void split_prod4(const float* x, const float* y, uint32_t (&w)[2][2]) {
        float p[4], q[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            p[k] = y ? x[k] * y[k] : x[k];
            q[k] = y ? y[k] : 1.0f;
        }
        const uint32_t h0 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[0], p[1]}, f16x2));
        const uint32_t h1 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[2], p[3]}, f16x2));
        uint32_t l0, l1;
        asm("v_fma_mixlo_f16 %0, %2, %6, -%10 op_sel_hi:[0,0,1]\n\t"
            "v_fma_mixhi_f16 %0, %3, %7, -%10 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
            "v_fma_mixlo_f16 %1, %4, %8, -%11 op_sel_hi:[0,0,1]\n\t"
            "v_fma_mixhi_f16 %1, %5, %9, -%11 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
            "s_nop 1"
            : "=&v"(l0), "=&v"(l1)
            : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]), "v"(h0),
              "v"(h1));
        w[0][0] = h0;
        w[0][1] = h1;
        w[1][0] = l0;
        w[1][1] = l1;
    }
    // split of x * s: h = fp16(x s), l = fp16(fma(x, s, -h)) (the residual
    // x s - h is exact in FP32 when s is a power of two times a float that
    // keeps x s in range, and fma computes it in one rounding otherwise)
    template <int N>
    static __device__ __forceinline__ void split_scaled(const float* v, float s, uint32_t (&w)[2][N / 2]) {
#pragma unroll
        for (int k = 0; k < N / 2; k++) {
            const f32x2 y = {v[2 * k] * s, v[2 * k + 1] * s};
            const f16x2 h = __builtin_convertvector(y, f16x2);
            const f32x2 r = {fmaf(v[2 * k], s, -(float)h[0]), fmaf(v[2 * k + 1], s, -(float)h[1])};
            const f16x2 l = __builtin_convertvector(r, f16x2);
            w[0][k] = __builtin_bit_cast(uint32_t, h);
            w[1][k] = __builtin_bit_cast(uint32_t, l);
        }
    }
    // c + a.b from the three products above the split's own error: with
    // a = ah + al + ea, |al| <= 2^-12 |a|, |ea| <= 2^-23 |a| (and the same for
    // b), the dropped al.bl is at most 2^-24 |a b|, below ea.b and a.eb
    static __device__ __forceinline__ f32x4 mma(const Op& a, const Op& b, f32x4 c) {
        c = mfma_f16(a.p[1], b.p[0], c);
        c = mfma_f16(a.p[0], b.p[1], c);
        c = mfma_f16(a.p[0], b.p[0], c);
        return c;
    }
    // The tap the fp16 pair represents exactly (the operand split of
    // tap(k) * 2^14 reproduces it), divided back by 2^14.
    static __device__ __forceinline__ float tap_value(int k) {
        const float x = tap(k) * kTapScale;
        const _Float16 h = (_Float16)x;
        const _Float16 l = (_Float16)(x - (float)h);
        return ((float)h + (float)l) * (1.f / kTapScale);
    }
};

// Six wave sums at once, in FP32, by a fixed butterfly of v_add_f32_dpp
// (x plus the value a DPP control brings from another lane): quad_perm
// [1,0,3,2] and [2,3,0,1] sum the quads, row_half_mirror and row_mirror the
// rows of 16 lanes; row_bcast:15 adds row 0 into row 1 and row 2 into row 3,
// row_bcast:31 row 1 into row 3 (rows outside a step's row mask keep their
// value). Lane 63 ends with ((r3 + r2) + (r1 + r0)), the same order every
// time. The six chains are interleaved, so that every DPP read comes six
// instructions after the write of its source (two wait states are needed;
// s_nop 1 covers the writes before the block).
__device__ __forceinline__ void wave_sums6(float (&x)[6]) {
    asm volatile(
        "s_nop 1\n\t"
        "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]));
}

// Orders this wave's LDS accesses before and after (the wave's lanes exchange
// data through LDS; no other wave touches the region).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename ST>
struct Load4;
template <>
struct Load4<float> {
    static __device__ __forceinline__ void run(const float* p, float v[4]) {
        const float4 a = *reinterpret_cast<const float4*>(p);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    }
};
template <>
struct Load4<__half> {
    static __device__ __forceinline__ void run(const __half* p, float v[4]) {
        const uint2 u = *reinterpret_cast<const uint2*>(p);
        const float2 f = __half22float2(*reinterpret_cast<const __half2*>(&u.x));
        const float2 g = __half22float2(*reinterpret_cast<const __half2*>(&u.y));
        v[0] = f.x; v[1] = f.y; v[2] = g.x; v[3] = g.y;
    }
};

// Byte offset of element x of row y of a plane (planes are far below 4 GiB),
// and the element at a byte offset from a plane base: the base stays in
// scalar registers and each load takes one 32-bit vector offset.
template <typename ST>
__device__ __forceinline__ uint32_t plane_off(int y, int64_t pitch, int x) {
    return ((uint32_t)y * (uint32_t)pitch + (uint32_t)x) * (uint32_t)sizeof(ST);
}
template <typename ST>
__device__ __forceinline__ const ST* at(const ST* base, uint32_t byte_off) {
    return reinterpret_cast<const ST*>(reinterpret_cast<const uint8_t*>(base) + byte_off);
}

// A wave's columns: two strips of 16 output columns, whose input is three
// windows of 16 columns. kMxWaves waves cover a tile's 64 columns.
constexpr int kMxWaves = kMxTile / 32;
constexpr int kRawPitch = 72;  // rows 8 banks apart

// Shared memory of one workgroup, for a split into NP parts; HS waves share
// the rows of each 32 columns.
template <int NP, int HS>
struct MxLds {
    // ring[wave][strip][moment][part][lane]: the last block's row-pass results,
    // rows 4g .. 4g + 3 of column j, as the row pass leaves them in lane (g, j)
    // and as the same lane's operand of the column pass takes them: registers
    // put aside, read by the lane that wrote them
    u32x2 ring[kMxWaves * HS][2][4][NP][64];
    // raw[wave][image][row]: the centred samples a and b, from the lanes that
    // hold a row of four columns to those that hold a pixel's maps (see RawAt)
    float raw[kMxWaves * HS][2][8][kRawPitch];
    double red[2][kMxWaves][kFeat];  // wave sums of the tile's upper and lower half
    float rowf[kMxTileH];  // renormalisation factor of the tile's output rows
    float cum[18];      // cumulative taps, as the split represents them
};

// Places of the samples in a wave's raw, in floats. The maps of 16 output rows
// need the last 8 rows of one input block and the first 8 of the next. A row
// holds 48 floats of the former, which the next block's maps read (columns
// 0 .. 7 and 16 .. 23 in one of two places by the block's parity), and 24 of the
// latter (column c at c % 24); the places keep the reads of rows 0 and 4 apart
// in the banks. A wave's
// LDS accesses are done in order: a strip's samples are read after the first
// rows of its last window are written and before that window's last rows, which
// may take the place of the block before's. (Read again from global memory, 8 to
// 24 rows after the row pass read them, they missed the L2, where 32 columns of
// 16 waves per CU do not stay that long: 240 1080p pairs took 11.9 ms.)
struct RawAt {
    int put[3];  // of this lane's four columns of window v
    int get[2];  // of row 4g, column j of strip q
    int mput[2], mget;  // 8 in the lanes whose place alternates: of put[0], put[1], of get
    __device__ __forceinline__ void init(int g, int j) {
        const int row = (j & 7) * kRawPitch;
        const bool next = j >= 8;  // this lane's rows are for the next block's maps
        put[0] = row + (next ? 0 : 48) + 4 * (g & 1);
        put[1] = row + (next ? 16 : 56) + 4 * g;
        put[2] = row + (next ? 40 : 48) + 4 * (g & 1);
        const int top = 4 * (g & 1) * kRawPitch;
        get[0] = top + (g < 2 ? (j < 8 ? j : 8 + j) : 48 + j);
        get[1] = top + (g < 2 ? (j < 8 ? 24 + j : 32 + j) : (j < 8 ? 64 + j : 40 + j));
        mput[0] = next ? 8 : 0;
        mput[1] = next && g >= 2 ? 8 : 0;
        mget = g < 2 && j < 8 ? 8 : 0;
    }
};

// Geometry of one tile, the same for every channel.
struct TileGeo {
    int W, H, x0, y0, g, j, wave;
    int xw;      // first output column of this wave
    int wcol;    // the wave's place in the tile: columns 32 wcol .. 32 wcol + 31
    int h_lo, h_hi;  // halves of the tile's rows that this wave takes
    int64_t pitch, pe;
};

// Taps of a split as operands. An operand's eight values of a lane are four of
// each of two windows of 16 input columns (row pass, B), or of two blocks of 16
// input rows (column pass, A): column or row 4g + e % 4 of either (the order in
// K is free, as long as both sides follow it). op[0] has the first window, or
// the older block, in elements 0 .. 3 and the second in 4 .. 7; op[1] the other
// way round.
template <typename SP>
struct MxTaps {
    typename SP::Op op[2];
};
template <typename SP>
__device__ __forceinline__ MxTaps<SP> tap_operands(int g, int j) {
    constexpr int NP = SP::kParts;
    MxTaps<SP> G;
#pragma unroll
    for (int v = 0; v < 2; v++) {
        float tv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 16 * v + 4 * g + e - j;
            tv[e] = (k >= 0 && k <= 16) ? SP::tap_value(k) * SP::kTapScale : 0.f;
        }
        uint32_t w[NP][2];
        SP::template split<4>(tv, w);
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                G.op[0].p[p][2 * v + k] = w[p][k];
                G.op[1].p[p][2 * (1 - v) + k] = w[p][k];
            }
    }
    return G;
}

// Channels c_lo .. c_hi - 1 of this wave's part of one tile; leaves their wave
// sums in red[half][wcol] (6 per channel, at 6 c).
//
// EDGE is false for tiles whose 80 x 144 input region lies inside the image:
// no element is masked, every output pixel is in the image and every
// renormalisation total is the full sum of the taps, so the factors fold into
// constants. Edge tiles clamp their loads into the image, give out-of-image
// elements the centre value (all four moments zero) and renormalise by the
// in-bounds taps of each output row and column.
//
// Scales: the row pass multiplies operands at the data scale (kScaleAB for a
// and b, kScaleDD^2 for (x1 - x2)^2, kScaleAB^2 kScaleQ for ab) by taps at
// kTapScale; its results are re-split at the data scale times the column
// factor (kmid); the column pass multiplies by the taps at kTapScale again,
// and edge tiles by the row factor.
template <typename SP, typename ST, int HS, bool EDGE>
__device__ __forceinline__ void mx_tile(MxLds<SP::kParts, HS>& L, const TileGeo& T, const MxTaps<SP>& G,
                                        const ST* base1, const ST* base2, const float* cum, int lane, int c_lo,
                                        int c_hi) {
    constexpr int NP = SP::kParts;
    const int W = T.W, H = T.H, g = T.g, j = T.j, wave = T.wave;
    const int64_t pitch = T.pitch;
    // scale of the means as the column pass leaves them, and what brings its
    // (a - b)^2 and ab to the square of it
    constexpr float kA = SP::kScaleAB, kS = kA * SP::kTapScale;
    constexpr float kE = kS * kS / (SP::kScaleDD * SP::kScaleDD * SP::kTapScale);
    constexpr float kQ = kS * kS / (SP::kScaleAB * SP::kScaleAB * SP::kScaleQ * SP::kTapScale);
    // Re-split scale of this lane's row-pass results (output columns xw + j and
    // xw + 16 + j): the renormalisation of their columns, in the interior that
    // of the rows as well (both by the full tap sum as the split represents it).
    const float inv_total = __builtin_amdgcn_rcpf(cum[17]);
    float kmid[2];
#pragma unroll
    for (int q = 0; q < 2; q++)
        kmid[q] = (EDGE ? __builtin_amdgcn_rcpf(tap_total(cum, T.xw + 16 * q + j, W)) : inv_total * inv_total) *
                  (1.f / SP::kTapScale);
    if (EDGE) {
        // table of the renormalisation of the tile's output rows (lane l: rows y0 + l + 64 q;
        // every wave writes the same values and reads its own)
#pragma unroll
        for (int q = 0; q < kMxTileH / 64; q++)
            L.rowf[lane + 64 * q] = __builtin_amdgcn_rcpf(tap_total(cum, min(T.y0 + lane + 64 * q, H - 1), H));
        wave_lds_sync();
    }
    // Work that can only add zeros is skipped on edge tiles: a wave whose
    // output columns all lie right of the image, a second strip that does, and
    // the row blocks below the last 16-row output block that holds an image
    // row (the last tile row of a scale often holds far fewer than 128 rows).
    // Skipping an addition of exact zeros leaves every sum bit for bit as it was.
    if (EDGE && T.xw >= W) {
        if (lane == 63)
            for (int hf = T.h_lo; hf < T.h_hi; hf++)
                for (int k = 0; k < kFeat; k++) L.red[hf][T.wcol][k] = 0.0;
        return;
    }
    const int nstrip = EDGE && T.xw + 16 >= W ? 1 : 2;
    constexpr int kMb = kMxTileH / 16 + 1;
    const int nmb = EDGE ? min(kMb, (min(H - T.y0, kMxTileH) + 15) / 16 + 1) : kMb;
    // The masks and selects of an edge tile are skipped, by a wave-uniform
    // branch, in the blocks that do not need them: when this wave's input
    // columns (xin) or output columns (xout) lie in the image, and so do the
    // block's rows, every mask bit is set and every select keeps its value.
    const bool xin = T.xw >= 8 && T.xw + 40 <= W, xout = T.xw + 32 <= W;
    // this lane's four input columns of window v, from xw - 8 + 16 v + 4g on: a
    // group that starts in the image is read in place, past W up to the row's
    // pitch (a multiple of 64 elements); a group wholly outside it is read at
    // column 0 and masked
    int xl[3], cmask = 0;  // cmask: bit 4 v + e, column e of window v lies in the image
#pragma unroll
    for (int v = 0; v < 3; v++) {
        const int xi = T.xw - 8 + 16 * v + 4 * g;
        const bool in = !EDGE || (xi >= 0 && xi < W);
        xl[v] = in ? xi : 0;
        if (EDGE) cmask |= in ? (int)((1u << min(W - xi, 4)) - 1u) << (4 * v) : 0;
    }

#pragma unroll 1
    for (int c = c_lo; c < c_hi; c++) {
        const ST* p1 = base1 + c * T.pe;
        const ST* p2 = base2 + c * T.pe;
        const int cxp = min(T.x0 + kMxTile / 2, W - 1), cyp = min(T.y0 + kMxTileH / 2, H - 1);
        // each image centred on its own value at the tile centre: a = x1 - cc,
        // b = x2 - cc2; the difference moment is then (a - b)^2, which stays
        // near 0 where the images differ by a locally constant offset, so
        // Vd = E[(a - b)^2] - (mu_a - mu_b)^2 does not cancel two large terms
        const float cc = ldf(p1 + (int64_t)cyp * pitch + cxp);
        const float cc2 = ldf(p2 + (int64_t)cyp * pitch + cxp);
        const float ccs = cc * SP::kScaleAB, ccs2 = cc2 * SP::kScaleAB;
        const float dc = cc - cc2;
        int mb = 4 * T.h_lo;
        RawAt R;
        R.init(g, j);
        float* const raw = &L.raw[wave][0][0][0];
        // The samples of a window are loaded while the one before it is worked
        // on (those of the last block's successor: that block's again).
        float n1[4], n2[4];
        auto load = [&](int b, int v) {
            const int y = T.y0 - 8 + 16 * min(b, nmb - 1) + j;
            const uint32_t ro = plane_off<ST>(EDGE ? min(max(y, 0), H - 1) : y, pitch, xl[v]);
            Load4<ST>::run(at(p1, ro), n1);
            Load4<ST>::run(at(p2, ro), n2);
        };
        load(mb, 0);
#pragma unroll 1
        for (int hf = T.h_lo; hf < T.h_hi; hf++) {
            float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            const int mb_end = min(nmb, 4 * hf + 5);
#pragma unroll 1
            for (; mb < mb_end; mb++) {
                const int ob = mb - 1;  // output rows y0 + 16 ob .. +15, from input blocks ob and mb
                const bool out = mb > 4 * T.h_lo;
                // ---- row pass of input rows y0 - 8 + 16 mb .. +15; this lane: row j
                const int yr = T.y0 - 8 + 16 * mb + j;
                const bool masks = EDGE && !(xin && T.y0 - 8 + 16 * mb >= 0 && T.y0 + 8 + 16 * mb <= H);
                const int odd = mb & 1 ? -1 : 0;
                const int put[3] = {R.put[0] + (odd & R.mput[0]), R.put[1] + (odd & R.mput[1]), R.put[2]};
                const int get[2] = {R.get[0] + (~odd & R.mget), R.get[1] + (~odd & R.mget)};
                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                typename SP::Op A[4];  // window v in half v & 1
#pragma unroll
                for (int v = 0; v < 3; v++) {
                    if (EDGE && v > nstrip) break;
                    float s1[4], s2[4];
                    {
                        if (masks) {
                            // one vector load per image for every lane: the
                            // row is clamped into the image and an element
                            // outside it takes the centre values cc and cc2,
                            // so that all four of its moments are exactly zero
                            // (ccs = cc kScaleAB is exact: the scale is a
                            // power of two)
                            const bool row_ok = yr >= 0 && yr < H;
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const bool in = row_ok && ((cmask >> (4 * v + e)) & 1);
                                n1[e] = in ? n1[e] : cc;
                                n2[e] = in ? n2[e] : cc2;
                            }
                        }
                        // the moments as products of two factors: a, b, dd dd, (a kScaleQ) b
                        float a[4], b[4], dd[4], aq[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            a[e] = fmaf(n1[e], SP::kScaleAB, -ccs);
                            b[e] = fmaf(n2[e], SP::kScaleAB, -ccs2);
                            dd[e] = (a[e] - b[e]) * (SP::kScaleDD / SP::kScaleAB);
                            aq[e] = a[e] * SP::kScaleQ;
                        }
                        if (v < nstrip) load(mb, v + 1 < 3 ? v + 1 : 0);
                        else load(mb + 1, 0);
                        // samples to the lanes of their pixels
                        auto store = [&] {
                            *reinterpret_cast<f32x4*>(raw + put[v]) = f32x4{a[0], a[1], a[2], a[3]};
                            *reinterpret_cast<f32x4*>(raw + put[v] + 8 * kRawPitch) = f32x4{b[0], b[1], b[2], b[3]};
                        };
                        if (v == 0) {
                            if (g >= 2) store();
                        } else {
                            if (j < 8 && (v == 1 || g < 2)) store();
                            wave_lds_sync();
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                s1[r] = raw[get[v - 1] + r * kRawPitch];
                                s2[r] = raw[get[v - 1] + r * kRawPitch + 8 * kRawPitch];
                            }
                            wave_lds_sync();
                            if (j >= 8 && (v == 1 || g < 2)) store();
                        }
                        const float* fx[4] = {a, b, dd, aq};
                        const float* fy[4] = {nullptr, nullptr, dd, b};
#pragma unroll
                        for (int m = 0; m < 4; m++) {
                            uint32_t w[NP][2];
                            SP::split_prod4(fx[m], fy[m], w);
#pragma unroll
                            for (int p = 0; p < NP; p++) {
                                A[m].p[p][2 * (v & 1)] = w[p][0];
                                A[m].p[p][2 * (v & 1) + 1] = w[p][1];
                            }
                        }
                    }
                    if (v == 0) continue;
                    const int q = v - 1;  // the strip that is complete
                    // Lane (g, j) holds rows 4g .. 4g+3 of the block, column j
                    // of the strip: half of its operand of the column pass as
                    // it stands; the other half is the block before, put aside
                    // in LDS (on a tile's first block, whatever was there: the
                    // products are not used).
                    f32x4 o[4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const f32x4 hr = SP::mma(A[m], G.op[q], z);
                        const float rv[4] = {hr[0], hr[1], hr[2], hr[3]};
                        uint32_t w[NP][2];
                        SP::template split_scaled<4>(rv, kmid[q], w);
                        typename SP::Op B;
#pragma unroll
                        for (int p = 0; p < NP; p++) {
                            // volatile: two reads in one instruction would
                            // need their halves moved into the operands
                            auto* r = (volatile __attribute__((address_space(3))) u32x2*)&L.ring[wave][q][m][p][lane];
                            const u32x2 old = *r;
                            B.p[p] = u32x4{old[0], old[1], w[p][0], w[p][1]};
                            *r = u32x2{w[p][0], w[p][1]};
                        }
                        o[m] = SP::mma(G.op[0], B, z);
                    }
                    if (!out) continue;
                    // ---- maps of this lane's output pixels: rows y0 + 16 ob + 4g + r, column xo
                    // (outside the image, a pixel adds zero through the selects
                    // on ok, which also discard the NaN that its zero
                    // renormalisation total gives)
                    const int xo = T.xw + 16 * q + j;
                    if (EDGE) {
                        const float4 rf = *reinterpret_cast<const float4*>(&L.rowf[16 * ob + 4 * g]);
                        const float f[4] = {rf.x, rf.y, rf.z, rf.w};
#pragma unroll
                        for (int m = 0; m < 4; m++)
#pragma unroll
                            for (int r = 0; r < 4; r++) o[m][r] *= f[r];
                    }
                    const int yo = T.y0 + 16 * ob + 4 * g;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        // SSIM: d = (Vd + md^2 num) / (Vd + num) with md the difference
                        // of the two means, Vd = var(x1 - x2), num = 2 cov + C2
                        // (src/ssimu2/score.hpp:141-148); mu1, mu2 are the centred
                        // means, so md = mu1 - mu2 + (cc - cc2). The means stay at
                        // their scale kS, and Vd and num at kS^2, which their
                        // quotient does not see: a power of two, so that every
                        // product is what it would be without it.
                        const float mu1 = o[0][r], mu2 = o[1][r];
                        const float mdc = mu1 - mu2;
                        const float vd = fmaf(o[2][r], kE, -(mdc * mdc));
                        const float md = fmaf(mdc, 1.f / kS, dc);
                        const float md2 = md * md;
                        const float num_s = fmaf(2.f, fmaf(o[3][r], kQ, -(mu1 * mu2)), 0.0009f * kS * kS);
                        const float n_s = fmaf(md2, num_s, vd);
                        const float den = vd + num_s;
                        // edge ratio (src/ssimu2/score.hpp:150-154)
                        const float fa = fmaf(fabsf(fmaf(mu1, -kA / kS, s1[r])), 1.f / kA, 1.f);
                        const float fb = fmaf(fabsf(fmaf(mu2, -kA / kS, s2[r])), 1.f / kA, 1.f);
                        // one reciprocal for both quotients: d = n / den and
                        // (fb - fa) / fa = (fb - fa) den / (den fa); fb - fa is
                        // exactly 0 for identical inputs, so both maps stay 0
                        const float rr = __builtin_amdgcn_rcpf(den * fa);
                        float d = (n_s * fa) * rr;
                        const float ev = ((fb - fa) * den) * rr;
                        float art = fmaxf(ev, 0.f), det = fmaxf(-ev, 0.f);
                        d = fmaxf(d, 0.f);
                        if (EDGE && !(xout && T.y0 + 16 * ob + 16 <= H)) {
                            const bool ok = xo < W && yo + r < H;
                            d = ok ? d : 0.f;
                            art = ok ? art : 0.f;
                            det = ok ? det : 0.f;
                        }
                        const float d2 = d * d, a2 = art * art, t2 = det * det;
                        acc[0] += d;
                        acc[1] = fmaf(d2, d2, acc[1]);
                        acc[2] += art;
                        acc[3] = fmaf(a2, a2, acc[3]);
                        acc[4] += det;
                        acc[5] = fmaf(t2, t2, acc[5]);
                    }
                }
            }
            // wave sums of this channel and half by the DPP butterfly (no LDS,
            // no lane permutes through it); the per-lane sums cover 32 pixels,
            // the wave sum 2,048, and a tile's four wave sums and the tiles
            // are added in FP64
            wave_sums6(acc);
            if (lane == 63) {
#pragma unroll
                for (int k = 0; k < 6; k++) L.red[hf][T.wcol][c * 6 + k] = (double)acc[k];
            }
        }
    }
}

}  // namespace

// Occupancy: the two-part split fits 3 waves per SIMD (13.1 KB of LDS per wave,
// at most 168 VGPRs, none spilled), the three-part split 2 (17.2 KB). 46 to 61
// SGPRs of either are kept in lanes of vector registers.
//
// HS: 1, a wave takes all rows of its 32 columns (workgroups of two waves); 2,
// half of them (four waves, 80 input rows for 64 instead of 144 for 128), for
// launches of few tiles (map_split). csplit: 1, a workgroup takes the three channels of a
// tile; 3, one channel (work item w: tile w / 3, channel w % 3). A wave sum
// covers one channel of one half of 32 columns either way, so every split gives
// the same partials bit for bit.
//
// With HS = 2 the first nsmall workgroups take the FP64 tiles of this plane
// storage, one channel of one tile each.
template <int NP, int HS>
union MapLds {
    MxLds<NP, HS> mx;
};
template <int NP>
union MapLds<NP, 2> {
    MxLds<NP, 2> mx;
    SmallLds small;
};
template <typename ST, typename SP, int HS>
__global__ __launch_bounds__(64 * kMxWaves * HS, SP::kParts == 2 ? 3 : 2) void map_mx_kernel(const PairDev* __restrict__ pairs,
                                                        const int32_t* __restrict__ order_seg,
                                                        const int32_t* __restrict__ order_start,
                                                        const BatchHdr* __restrict__ hdr,
                                                        const uint8_t* __restrict__ arena,
                                                        double* __restrict__ partials, int csplit,
                                                        int nsmall) {
    constexpr int TS = kMxTile;
    constexpr int grp = map_group(0, sizeof(ST) == 2, SP::kParts == 3);
    __shared__ MapLds<SP::kParts, HS> lds;
    if constexpr (HS == 2) {
        if ((int)blockIdx.x < nsmall) {
            map_small_tile<ST>(lds.small, pairs, order_seg, order_start, hdr, arena, partials, blockIdx.x);
            return;
        }
    }
    MxLds<SP::kParts, HS>& L = lds.mx;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, j = lane & 15;
    if (tid == 0) {
        float a = 0.f;
        L.cum[0] = 0.f;
        for (int k = 0; k < 17; k++) {
            a += SP::tap_value(k);
            L.cum[k + 1] = a;
        }
    }
    __syncthreads();

    const MxTaps<SP> G = tap_operands<SP>(g, j);

    int seg_lo = 0, t_begin = 0;
#pragma unroll
    for (int q = 0; q < grp; q++) {
        seg_lo += hdr->nseg[q];
        t_begin += hdr->tiles[q];
    }
    const int seg_hi = seg_lo + hdr->nseg[grp] - 1;
    const int t_end = t_begin + hdr->tiles[grp];
    // A grid of one workgroup per work item (or more) numbers its workgroups
    // with xcd_block, so that the workgroups of one XCD hold one contiguous
    // range of tiles. A smaller, persistent grid takes its work items from the
    // per-XCD dynamic queue.
    const int nwg = gridDim.x - nsmall;
    const int ntl = t_end - t_begin;
    const int nwork = ntl * csplit;
    const bool persistent = nwg < nwork;
    int32_t* queue = const_cast<int32_t*>(hdr->queue[grp]);
    __shared__ int s_tile;
    // (with more workgroups than work items, item floor(v n / nwg) of virtual
    // workgroup v, so that every XCD still gets work)
    const int vb = xcd_block(blockIdx.x - nsmall, nwg);
    int next = (int)(((int64_t)vb * nwork) / nwg);
    const int w_hi = (int)(((int64_t)(vb + 1) * nwork) / nwg);
    for (;;) {
        int w;
        if (persistent) {
            if (tid == 0) s_tile = queue_next(queue, nwork);
            __syncthreads();
            w = s_tile;  // read by every thread before the tile's closing barrier
            if (w < 0) break;
        } else {
            if (next >= w_hi) break;
            w = next++;
        }
        const int tq = w / csplit, part = w - tq * csplit;
        const int t = t_begin + tq;
        const int c_lo = csplit == 1 ? 0 : part, c_hi = csplit == 1 ? 3 : part + 1;
        int lo = seg_lo, hi = seg_hi;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (order_start[mid] <= t) lo = mid;
            else hi = mid - 1;
        }
        const int seg = order_seg[lo];
        const int pair = seg / kScales, s = seg - pair * kScales;
        const PairDev& P = pairs[pair];
        TileGeo T;
        T.W = P.sw[s];
        T.H = P.sh[s];
        T.pitch = P.pitch[s];
        T.pe = P.plane_elems[s];
        const int ntx = (T.W + TS - 1) / TS;
        const int local = t - order_start[lo];
        const int ty = local / ntx, tx = local - ty * ntx;
        T.x0 = tx * TS;
        T.y0 = ty * kMxTileH;
        T.g = g;
        T.j = j;
        T.wave = wave;
        T.wcol = wave % kMxWaves;
        T.xw = T.x0 + 32 * T.wcol;
        T.h_lo = HS == 1 ? 0 : wave / kMxWaves;
        T.h_hi = HS == 1 ? 2 : T.h_lo + 1;
        const ST* base1 = reinterpret_cast<const ST*>(arena + P.arena_off + P.scale_off[s]);
        const ST* base2 = reinterpret_cast<const ST*>(arena + P.arena_off + P.img_bytes + P.scale_off[s]);
        // the 80 x 144 input region in the image: no masks, constant renormalisation
        const bool interior = T.x0 >= 8 && T.x0 + kMxTile + 8 <= T.W && T.y0 >= 8 && T.y0 + kMxTileH + 8 <= T.H;
        if (interior) mx_tile<SP, ST, HS, false>(L, T, G, base1, base2, L.cum, lane, c_lo, c_hi);
        else mx_tile<SP, ST, HS, true>(L, T, G, base1, base2, L.cum, lane, c_lo, c_hi);

        __syncthreads();
        if (tid >= 6 * c_lo && tid < 6 * c_hi) {
            const double sum = ((L.red[0][0][tid] + L.red[0][1][tid]) + L.red[1][0][tid]) + L.red[1][1][tid];
            partials[(int64_t)t * kFeat + tid] = sum;
        }
        __syncthreads();
    }
}

// The FP64 tiles by themselves, for grids of a fixed size (capture, persistent).
template <typename ST>
__global__ __launch_bounds__(256) void map_small_kernel(const PairDev* __restrict__ pairs,
                                                        const int32_t* __restrict__ order_seg,
                                                        const int32_t* __restrict__ order_start,
                                                        const BatchHdr* __restrict__ hdr,
                                                        const uint8_t* __restrict__ arena,
                                                        double* __restrict__ partials) {
    __shared__ SmallLds L;
    const int n = 3 * hdr->tiles[map_group(1, sizeof(ST) == 2)];
    for (int item = blockIdx.x; item < n; item += gridDim.x) {
        map_small_tile<ST>(L, pairs, order_seg, order_start, hdr, arena, partials, item);
        __syncthreads();
    }
}

hipError_t launch_map_small(bool half, int grid, const PairDev* pairs, const int32_t* order_seg,
                            const int32_t* order_start, const BatchHdr* hdr, const void* arena, double* partials,
                            hipStream_t st) {
    const uint8_t* a = reinterpret_cast<const uint8_t*>(arena);
    if (half) map_small_kernel<__half><<<grid, 256, 0, st>>>(pairs, order_seg, order_start, hdr, a, partials);
    else map_small_kernel<float><<<grid, 256, 0, st>>>(pairs, order_seg, order_start, hdr, a, partials);
    return hipGetLastError();
}

namespace {
template <typename ST, typename SP>
void launch_mx(int rows, int grid, int nsmall, const PairDev* pairs, const int32_t* order_seg,
               const int32_t* order_start, const BatchHdr* hdr, const uint8_t* arena, double* partials, int csplit,
               hipStream_t st) {
    if (rows == 2)
        map_mx_kernel<ST, SP, 2><<<grid + nsmall, 128 * kMxWaves, 0, st>>>(pairs, order_seg, order_start, hdr, arena, partials, csplit, nsmall);
    else
        map_mx_kernel<ST, SP, 1><<<grid, 64 * kMxWaves, 0, st>>>(pairs, order_seg, order_start, hdr, arena, partials, csplit, 0);
}
}  // namespace

hipError_t launch_map_mx(bool half, bool exact, int rows, int grid, int nsmall, const PairDev* pairs,
                         const int32_t* order_seg, const int32_t* order_start, const BatchHdr* hdr, const void* arena,
                         double* partials, int csplit, hipStream_t st) {
    if ((csplit != 1 && csplit != 3) || (rows != 1 && rows != 2) || (rows == 1 && nsmall)) return hipErrorInvalidValue;
    const uint8_t* a = reinterpret_cast<const uint8_t*>(arena);
    // float RGB input may hold any value: the exact split; every other format
    // gives bounded XYB values: the scaled fp16 split
    auto* run = exact ? (half ? launch_mx<__half, SplitBf16x3> : launch_mx<float, SplitBf16x3>)
                      : (half ? launch_mx<__half, SplitF16x2> : launch_mx<float, SplitF16x2>);
    run(rows, grid, nsmall, pairs, order_seg, order_start, hdr, a, partials, csplit, st);
    return hipGetLastError();
}

}  // namespace vship
