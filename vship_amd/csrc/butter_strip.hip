// Butteraugli's blurs on the gfx950 matrix cores, fused with what surrounds
// them: opsin, low, mid and high of butter.hip's stage list, for inputs of
// ordinary range.
//
// A workgroup takes a strip of 32 columns by th rows of one pair and scale,
// and one wave of it blurs each plane that the stage's point operations need
// together (both images, all channels). The wave streams down the strip in
// blocks of 16 rows, everything in registers:
//
//   row pass     Hr(16 rows x 16 cols) = In(16 x 32 input cols) . G(32 x 16)
//   column pass  Out(16 rows x 16 cols) = G'(16 x 32 input rows) . Hr(32 x 16)
//
// on v_mfma_f32_16x16x32_f16, G being the band of taps. A lane loads the
// eight consecutive samples that are its operand straight from the plane, and
// the row pass leaves four rows of one column in a lane, which are half of
// its operand of the column pass as they stand (an operand's order in K is
// free, as long as the taps follow it): no LDS and no barrier between load and
// result. The results of all planes meet in LDS, where 256 threads take two
// neighbouring pixels each through the point operations and write them as
// 8-byte pieces of whole rows.
//
// Operands are split into two fp16 parts x = h + l (h rounded towards zero,
// l to nearest), the products hh + hl + lh accumulate in FP32. A value keeps
// 22 to 23 significant bits, or an absolute error of 2^-25 where its low part
// is subnormal: linear RGB is therefore stored times 2^10, and the taps carry
// 2^14. fp16 ends at 65,504, and inputs are not bounded by nature (float RGB;
// chroma far outside the gamut next to its opposite, at a high intensity):
// the opsin stage checks every sample and every result against kLinMax and
// kXybMax, below which no later value leaves the range (XYB minus its low
// band is below 2 kXybMax, minus its middle band below 4 kXybMax = 32,768). A
// pair that fails, NaN included, is marked, and the engine scores it again
// with the general kernels.
#include <cmath>
#include <cstring>

#include <hip/hip_fp16.h>

#include "butter_dev.hpp"
#include "butter_strip.hpp"

namespace vship {
namespace bt {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kTapScale = 16384.0f;
constexpr float kLinMax = 32768.0f;  // of linear RGB times kLinScale
constexpr float kXybMax = 8192.0f;

// ---------------------------------------------------------------------------
// geometry of a strip blur of radius R
// ---------------------------------------------------------------------------
// Row pass: kGroups loads of 8 columns per lane; load q of a lane of group
// g = lane / 16 starts at column strip + col(q, g), and output block b
// (columns 16 b .. 16 b + 15) multiplies loads in(b, 0) .. in(b, kRowSteps - 1).
// Column pass: the ring holds kRing blocks of 16 rows, the first kRowOff rows
// above the output block.
template <int R>
struct Geo;
template <>
struct Geo<8> {
    // 16 + 2 * 8 = 32 columns and rows: one step each
    static constexpr int kGroups = 2, kRowSteps = 1, kRing = 2, kRowOff = 8, kRowOps = 1, kColOps = 1;
    static __host__ __device__ constexpr int col(int q, int g) { return (q ? 8 : -8) + 8 * g; }
    static __host__ __device__ constexpr int in(int b, int) { return b; }
    static __host__ __device__ constexpr int op(int, int) { return 0; }
};
template <>
struct Geo<9> {
    // 34 columns and rows: two steps, both blocks from the same 64 columns;
    // of the second step of the column pass only half has taps
    static constexpr int kGroups = 2, kRowSteps = 2, kRing = 3, kRowOff = 16, kRowOps = 4, kColOps = 2;
    static __host__ __device__ constexpr int col(int q, int g) { return (q ? 16 : -16) + 8 * g; }
    static __host__ __device__ constexpr int in(int, int s) { return s; }
    static __host__ __device__ constexpr int op(int b, int s) { return 2 * b + s; }
};
template <>
struct Geo<21> {
    // 58 columns and rows: two steps each. Block 0 reads columns -24 .. 39,
    // block 1 -8 .. 55, of which load 2 brings -8 .. 7 and 40 .. 55.
    static constexpr int kGroups = 3, kRowSteps = 2, kRing = 4, kRowOff = 24, kRowOps = 4, kColOps = 2;
    static __host__ __device__ constexpr int col(int q, int g) {
        return q == 1 ? 8 + 8 * g : (q == 2 && g < 2 ? 40 + 8 * g : -24 + 8 * g);
    }
    static __host__ __device__ constexpr int in(int b, int s) { return b + s; }
    static __host__ __device__ constexpr int op(int b, int s) { return 2 * b + s; }
};

// Tap index of element e of the row-pass operand of lane (g, j) in step s of
// block b, and of the column-pass operand in step s (elements 0..3 hold rows
// 4 g .. 4 g + 3 of ring block 2 s, elements 4..7 those of block 2 s + 1).
template <int R>
constexpr int row_tap(int b, int s, int g, int j, int e) {
    return Geo<R>::col(Geo<R>::in(b, s), g) + e - (16 * b + j) + R;
}
template <int R>
constexpr int col_tap(int s, int g, int j, int e) {
    return -Geo<R>::kRowOff + 16 * (2 * s + (e >> 2)) + 4 * g + (e & 3) - j + R;
}

// ---------------------------------------------------------------------------
// two-way fp16 split and its products
// ---------------------------------------------------------------------------
struct Op {
    u32x4 h, l;  // 8 values each
};

// x[0..7] -> h + l. The low parts are v_fma_mixlo/mixhi_f16 (x - h exactly,
// rounded once), written by inline assembly; the block ends with s_nop 1,
// since the compiler counts no wait states between inline assembly and a
// matrix instruction that reads its result.
__device__ __forceinline__ Op split8(const float (&x)[8]) {
    uint32_t h[4], l0, l1, l2, l3;
#pragma unroll
    for (int k = 0; k < 4; k++)
        h[k] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x[2 * k], x[2 * k + 1]));
    const float one = 1.0f;
    asm("v_fma_mixlo_f16 %0, %4, %12, -%13 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %5, %12, -%13 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, %6, %12, -%14 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %1, %7, %12, -%14 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %2, %8, %12, -%15 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %2, %9, %12, -%15 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %10, %12, -%16 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %11, %12, -%16 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 1"
        : "=&v"(l0), "=&v"(l1), "=&v"(l2), "=&v"(l3)
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(one),
          "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]));
    return {u32x4{h[0], h[1], h[2], h[3]}, u32x4{l0, l1, l2, l3}};
}

// half an operand: four values times s, by compiler code (they come from
// matrix instructions, whose wait states the compiler counts)
struct Half {
    u32x2 h, l;
};
__device__ __forceinline__ Half split4(f32x4 v, float s) {
    Half o;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const float a = v[2 * k] * s, b = v[2 * k + 1] * s;
        const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
        const f16x2 l = __builtin_convertvector((f32x2){a - (float)h[0], b - (float)h[1]}, f16x2);
        o.h[k] = __builtin_bit_cast(uint32_t, h);
        o.l[k] = __builtin_bit_cast(uint32_t, l);
    }
    return o;
}

__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}
__device__ __forceinline__ f32x4 mfma16(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0,
                                                 0);
}
// c + a . b; the dropped l l is at most 2^-22 of the product
__device__ __forceinline__ f32x4 mma(const Op& a, const Op& b, f32x4 c) {
    c = mfma32(a.l, b.h, c);
    c = mfma32(a.h, b.l, c);
    return mfma32(a.h, b.h, c);
}

// ---------------------------------------------------------------------------
// the stages: planes blurred together and their point operations
// ---------------------------------------------------------------------------
// Results of the planes at two neighbouring pixels, and the two pixels' place.
constexpr int kExPitch = 36;  // 4 rows of 36 floats start 16 banks apart
template <int P>
using Exchange = float[P][16][kExPitch];

struct Px {
    int row, col;  // in the block
    int g;         // element offset in a plane
    bool two;      // the second pixel lies in the image
};

__device__ __forceinline__ float2 at2(const float* base, int off) {
    return *reinterpret_cast<const float2*>(&at(const_cast<float*>(base), off));
}
__device__ __forceinline__ void put2(float* base, int off, const float (&v)[2]) {
    *reinterpret_cast<float2*>(&at(base, off)) = make_float2(v[0], v[1]);
}
template <int P>
__device__ __forceinline__ void take(const Exchange<P>& E, int p, const Px& X, float (&v)[2]) {
    const float2 t = *reinterpret_cast<const float2*>(&E[p][X.row][X.col]);
    v[0] = t.x;
    v[1] = t.y;
}

template <int P>
struct Centres {
    float v[P][2];
};
template <int P>
__device__ __forceinline__ void load_centres(Centres<P>& C, const Scale& S, int pair, int plane, int g) {
#pragma unroll
    for (int p = 0; p < P; p++) {
        const float2 t = at2(plane_u(S, pair, plane + p), g);
        C.v[p][0] = t.x;
        C.v[p][1] = t.y;
    }
}

// sigma 1.2 blur of linear RGB + opsin dynamics (colors.hpp:50-91): X and Y of
// both images, and the difference of the two Bs, all that the later stages
// need of it (they are linear in B)
struct OpsinStage {
    static constexpr int R = 8, kSig = SG_OPSIN, kPlanes = 6, kSrc = Q_LIN, kCentres = 6;
    static __device__ __forceinline__ void points(const Exchange<6>& E, const Px& X, const Centres<6>& C,
                                                  const Scale& S, int pair, const StripArgs& A) {
        float z[2][2];
        bool ok = true;
#pragma unroll
        for (int im = 0; im < 2; im++) {
            float bl[3][2], x[2], y[2];
#pragma unroll
            for (int c = 0; c < 3; c++) take<6>(E, 3 * im + c, X, bl[c]);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float* ctr[3] = {C.v[3 * im], C.v[3 * im + 1], C.v[3 * im + 2]};
                float b0, b1, b2, o0, o1, o2;
                opsin_absorbance(bl[0][k] * A.intensity, bl[1][k] * A.intensity, bl[2][k] * A.intensity, b0, b1, b2);
                opsin_absorbance(ctr[0][k] * A.intensity, ctr[1][k] * A.intensity, ctr[2][k] * A.intensity, o0, o1, o2);
                opsin_respond(b0, b1, b2, o0, o1, o2);
                x[k] = o0 - o1;
                y[k] = o0 + o1;
                z[im][k] = o2;
                // o0, o1 and o2 are positive, so the sums bound X, Y and B
                const bool in = fabsf(ctr[0][k]) <= kLinMax && fabsf(ctr[1][k]) <= kLinMax &&
                                fabsf(ctr[2][k]) <= kLinMax && y[k] <= kXybMax && o2 <= kXybMax;
                ok = ok && (in || (k == 1 && !X.two));
            }
            put2(plane_u(S, pair, Q_XY + 2 * im), X.g, x);
            put2(plane_u(S, pair, Q_XY + 2 * im + 1), X.g, y);
        }
        const float d[2] = {z[0][0] - z[1][0], z[0][1] - z[1][1]};
        put2(plane_u(S, pair, Q_DB), X.g, d);
        if (!ok) A.pairs[pair].general = 1;
    }
};

// sigma 7.156 blur: residual XYB - low band, and the L2 terms of the low
// bands as values (separatefrequencies.hpp:142-170, 3-13; simplerdiff.hpp:38-58)
struct LowStage {
    static constexpr int R = 21, kSig = SG_LOW, kPlanes = 5, kSrc = Q_XY, kCentres = 5;
    static __device__ __forceinline__ void points(const Exchange<5>& E, const Px& X, const Centres<5>& C,
                                                  const Scale& S, int pair, const StripArgs&) {
        float lf[5][2], dc[2];
#pragma unroll
        for (int p = 0; p < 5; p++) {
            take<5>(E, p, X, lf[p]);
            const float t[2] = {C.v[p][0] - lf[p][0], C.v[p][1] - lf[p][1]};
            put2(plane_u(S, pair, Q_T + p), X.g, t);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float dx = lf[0][k] - lf[2][k], dy = lf[1][k] - lf[3][k], db = lf[4][k] + -0.362267051518f * dy;
            const float vx = dx * 33.832837186260f, vy = dy * 14.458268100570f, vb = db * 49.87984651440f;
            dc[k] = 29.2353797994f * vx * vx;
            dc[k] += 0.844626970982f * vy * vy;
            dc[k] += 0.703646627719f * vb * vb;
        }
        put2(plane_u(S, pair, P_DCS), X.g, dc);
    }
};

// sigma 3.225 blur of the residual: middle bands after their range
// operations, as Malta differences and L2 terms; high residual, X's
// suppressed by Y's (separatefrequencies.hpp:160-189)
struct MidStage {
    static constexpr int R = 9, kSig = SG_MID, kPlanes = 5, kSrc = Q_T, kCentres = 4;
    static __device__ __forceinline__ void points(const Exchange<5>& E, const Px& X, const Centres<4>& C,
                                                  const Scale& S, int pair, const StripArgs& A) {
        float mf[5][2], hx[2][2], hy[2][2], ac[2], sx[2], sy[2];
#pragma unroll
        for (int p = 0; p < 5; p++) take<5>(E, p, X, mf[p]);
#pragma unroll
        for (int k = 0; k < 2; k++) {
#pragma unroll
            for (int im = 0; im < 2; im++) {
                hx[im][k] = C.v[2 * im][k] - mf[2 * im][k];
                const float yv = hy[im][k] = C.v[2 * im + 1][k] - mf[2 * im + 1][k];
                const float s = 0.653020556257f, yw = 46.0f;
                // hardware reciprocal (1 ulp) of a denominator of at least 46
                hx[im][k] *= s + (yw * (1.0f - s)) * __builtin_amdgcn_rcpf(yw + yv * yv);
            }
            const float x0 = remove_range(mf[0][k], 0.29f), x1 = remove_range(mf[2][k], 0.29f);
            const float y0 = amplify_range(mf[1][k], 0.1f), y1 = amplify_range(mf[3][k], 0.1f);
            const float dx = x0 - x1, dy = y0 - y1, db = mf[4][k];
            ac[k] = 2150.0f * dx * dx;
            ac[k] += 10.6195433239f * dy * dy;
            ac[k] += 16.2176043152f * db * db;
            sy[k] = malta_scaled_diff(y0, y1, A.diff.malta[4]);
            sx[k] = malta_scaled_diff(x0, x1, A.diff.malta[5]);
        }
#pragma unroll
        for (int im = 0; im < 2; im++) {
            put2(plane_u(S, pair, Q_HFR + 2 * im), X.g, hx[im]);
            put2(plane_u(S, pair, Q_HFR + 2 * im + 1), X.g, hy[im]);
        }
        put2(plane_u(S, pair, Q_SD + 4), X.g, sy);
        put2(plane_u(S, pair, Q_SD + 5), X.g, sx);
        put2(plane_u(S, pair, Q_ACM), X.g, ac);
    }
};

// sigma 1.564 blur of the high residual: high and ultra-high bands as Malta
// differences, L2 terms and mask inputs (separatefrequencies.hpp:117-140,
// 190-200; simplerdiff.hpp:60-101; maskPsycho.hpp:24-40)
struct HighStage {
    static constexpr int R = 8, kSig = SG_HIGH, kPlanes = 4, kSrc = Q_HFR, kCentres = 4;
    static __device__ __forceinline__ void points(const Exchange<4>& E, const Px& X, const Centres<4>& C,
                                                  const Scale& S, int pair, const StripArgs& A) {
        float hf[4][2], m[2][2], sd[4][2], ac[2];
#pragma unroll
        for (int p = 0; p < 4; p++) take<4>(E, p, X, hf[p]);
        const float2 acm = at2(plane_u(S, pair, Q_ACM), X.g);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            float h[4], u[4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                float hv = hf[p][k], uv = C.v[p][k];
                if (p & 1) {
                    hv = maximum_clamp(hv, 28.4691806922f);
                    uv -= hv;
                    uv = maximum_clamp(uv, 5.19175294647f);
                    uv *= 2.69313763794f;
                    hv *= 2.155f;
                    hv = amplify_range(hv, 0.132f);
                } else {
                    uv -= hv;
                    hv = remove_range(hv, 1.5f);
                    uv = remove_range(uv, 0.04f);
                }
                h[p] = hv;
                u[p] = uv;
            }
            sd[0][k] = malta_scaled_diff(u[1], u[3], A.diff.malta[0]);
            sd[1][k] = malta_scaled_diff(u[0], u[2], A.diff.malta[1]);
            sd[2][k] = malta_scaled_diff(h[1], h[3], A.diff.malta[2]);
            sd[3][k] = malta_scaled_diff(h[0], h[2], A.diff.malta[3]);
            ac[k] = k ? acm.y : acm.x;
            ac[k] += l2_asym(h[0], h[2], A.diff.asym_gt[0], A.diff.asym_lt[0]);
            ac[k] += l2_asym(h[1], h[3], A.diff.asym_gt[1], A.diff.asym_lt[1]);
            m[0][k] = mask_input(h[0], u[0], h[1], u[1]);
            m[1][k] = mask_input(h[2], u[2], h[3], u[3]);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) put2(plane_u(S, pair, Q_SD + t), X.g, sd[t]);
        put2(plane_u(S, pair, P_ACS), X.g, ac);
        put2(plane_u(S, pair, P_M0), X.g, m[0]);
        put2(plane_u(S, pair, P_M1), X.g, m[1]);
    }
};

// ---------------------------------------------------------------------------
// the strip kernel
// ---------------------------------------------------------------------------
template <class K>
__global__ __launch_bounds__(64 * K::kPlanes) void butter_strip_kernel(Scales SS, int npairs, int th,
                                                                       const StripTables* __restrict__ tab,
                                                                       StripArgs A) {
    constexpr int R = K::R;
    using G = Geo<R>;
    constexpr int kThreadsPx = 256;  // threads of the point operations
    __shared__ Exchange<K::kPlanes> ex[2];
    // scale, pair and strip of this workgroup
    const int nx0 = cdiv(SS.s[0].w, kStripW), ny0 = cdiv(SS.s[0].h, th);
    const int n0 = nx0 * ny0 * npairs;
    const bool half = (int)blockIdx.x >= n0;
    const Scale S = half ? SS.s[1] : SS.s[0];
    const TileIdx ti = half ? tile_of(blockIdx.x - n0, cdiv(S.w, kStripW), cdiv(S.h, th), npairs)
                            : tile_of(blockIdx.x, nx0, ny0, npairs);
    const int pair = ti.z, x0 = ti.x * kStripW, y0 = ti.y * th;
    const int w = S.w, h = S.h, pitch = S.pitch;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    const float* src = plane_u(S, pair, K::kSrc + wave);

    // this lane's columns: a load of 8 starts at a multiple of 8 and is read in
    // place if it starts in the image (past w up to the pitch, a multiple of
    // 64), at column 0 and masked otherwise
    int col[G::kGroups], cmask[G::kGroups];
#pragma unroll
    for (int q = 0; q < G::kGroups; q++) {
        const int c = x0 + G::col(q, g);
        const bool in = c >= 0 && c < w;
        col[q] = in ? c : 0;
        cmask[q] = in ? (int)((1u << min(w - c, 8)) - 1u) : 0;
    }
    const bool cols_in = x0 >= 24 && x0 + 56 <= w;  // every load of every lane lies in the image

    float v[G::kGroups][8];
    auto load = [&](int yb) {
        const int row = min(max(yb + j, 0), h - 1) * pitch;
#pragma unroll
        for (int q = 0; q < G::kGroups; q++) {
            const float4* p = reinterpret_cast<const float4*>(&at(const_cast<float*>(src), row + col[q]));
            const float4 a = p[0], b = p[1];
            v[q][0] = a.x; v[q][1] = a.y; v[q][2] = a.z; v[q][3] = a.w;
            v[q][4] = b.x; v[q][5] = b.y; v[q][6] = b.z; v[q][7] = b.w;
        }
    };
    load(y0 - G::kRowOff);

    Op rop[G::kRowOps], cop[G::kColOps];
    const u32x4* ops = reinterpret_cast<const u32x4*>(tab->op[K::kSig]);
#pragma unroll
    for (int i = 0; i < G::kRowOps; i++) rop[i] = {ops[(2 * i) * 64 + lane], ops[(2 * i + 1) * 64 + lane]};
#pragma unroll
    for (int i = 0; i < G::kColOps; i++)
        cop[i] = {ops[(2 * (G::kRowOps + i)) * 64 + lane], ops[(2 * (G::kRowOps + i) + 1) * 64 + lane]};
    const Taps* T = &tab->taps[K::kSig];
    const float full = 1.0f / T->cum[2 * R + 1] * (1.0f / kTapScale);
    float kcol[2];
#pragma unroll
    for (int b = 0; b < 2; b++)
        kcol[b] = cols_in ? full : inv_total<R>(T, min(x0 + 16 * b + j, w - 1), w) * (1.0f / kTapScale);

    // the two pixels of this thread in the point operations
    Px X;
    X.row = threadIdx.x >> 4;
    X.col = 2 * (threadIdx.x & 15);
    const int gx = x0 + X.col;
    X.two = gx + 1 < w;

    Half ring[2][G::kRing];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int k = 0; k < G::kRing; k++) ring[b][k] = {u32x2{0, 0}, u32x2{0, 0}};
    const int nout = cdiv(min(th, h - y0), 16);
    const int nblk = nout + G::kRing - 1;
#pragma unroll 1
    for (int i = 0; i < nblk; i++) {
        const int yb = y0 - G::kRowOff + 16 * i;
        if (!(cols_in && yb >= 0 && yb + 16 <= h)) {
            const bool row_in = yb + j >= 0 && yb + j < h;
#pragma unroll
            for (int q = 0; q < G::kGroups; q++)
#pragma unroll
                for (int e = 0; e < 8; e++) v[q][e] = row_in && ((cmask[q] >> e) & 1) ? v[q][e] : 0.0f;
        }
        Op a[G::kGroups];
#pragma unroll
        for (int q = 0; q < G::kGroups; q++) a[q] = split8(v[q]);
        // all splits before the first matrix instruction: inline assembly is
        // not checked against matrix instructions in flight
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < nblk) load(yb + 16);
#pragma unroll
        for (int b = 0; b < 2; b++) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < G::kRowSteps; s++) acc = mma(a[G::in(b, s)], rop[G::op(b, s)], acc);
#pragma unroll
            for (int k = 0; k + 1 < G::kRing; k++) ring[b][k] = ring[b][k + 1];
            ring[b][G::kRing - 1] = split4(acc, kcol[b]);
        }
        if (i < G::kRing - 1) continue;

        const int ob = i - (G::kRing - 1), yo = y0 + 16 * ob;
        const int gy = yo + X.row;
        const bool active = threadIdx.x < kThreadsPx && gx < w && gy < h;
        X.g = gy * pitch + gx;
        Centres<K::kCentres> C;
        if (active) load_centres<K::kCentres>(C, S, pair, K::kSrc, X.g);
        float krow[4];
        if (yo >= R && yo + 16 + R <= h) {
#pragma unroll
            for (int r = 0; r < 4; r++) krow[r] = full;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                krow[r] = inv_total<R>(T, min(yo + 4 * g + r, h - 1), h) * (1.0f / kTapScale);
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < G::kColOps; s++) {
                const Half& p = ring[b][2 * s];
                if (2 * s + 1 < G::kRing) {
                    const Half& q = ring[b][2 * s + 1 < G::kRing ? 2 * s + 1 : 0];
                    o = mma(cop[s], {u32x4{p.h[0], p.h[1], q.h[0], q.h[1]}, u32x4{p.l[0], p.l[1], q.l[0], q.l[1]}}, o);
                } else {
                    const u32x2 th2 = {cop[s].h[0], cop[s].h[1]}, tl2 = {cop[s].l[0], cop[s].l[1]};
                    o = mfma16(tl2, p.h, o);
                    o = mfma16(th2, p.l, o);
                    o = mfma16(th2, p.h, o);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) ex[ob & 1][wave][4 * g + r][16 * b + j] = o[r] * krow[r];
        }
        // one barrier per block: a wave writes a buffer again only after the
        // barrier of the block between, which every reader of it has reached
        __syncthreads();
        if (active) K::points(ex[ob & 1], X, C, S, pair, A);
    }
}

template <class K>
void launch(const Scales& SS, int n, int th, const StripTables* tab, const StripArgs& A, hipStream_t st) {
    const int64_t wgs = (int64_t)n * (cdiv(SS.s[0].w, kStripW) * cdiv(SS.s[0].h, th) +
                                      cdiv(SS.s[1].w, kStripW) * cdiv(SS.s[1].h, th));
    butter_strip_kernel<K><<<dim3((unsigned)wgs), dim3(64 * K::kPlanes), 0, st>>>(SS, n, th, tab, A);
}

template <int R>
void fill(StripTables& T, int sig) {
    using G = Geo<R>;
    double g[2 * R + 1], tot = 0.0, run = 0.0;
    uint16_t hi[2 * R + 1], lo[2 * R + 1];
    for (int k = -R; k <= R; k++) tot += g[k + R] = std::exp(-(double)k * k / (2.0 * kSigma[sig] * kSigma[sig]));
    for (int k = 0; k <= 2 * R; k++) {
        // the value the fp16 pair represents, and the sums of those values
        const float x = (float)(g[k] / tot) * kTapScale;
        const __half a = __float2half_rn(x), b = __float2half_rn(x - __half2float(a));
        hi[k] = __half_raw(a).x;
        lo[k] = __half_raw(b).x;
        T.taps[sig].g[k] = (__half2float(a) + __half2float(b)) / kTapScale;
        T.taps[sig].cum[k] = (float)run;
        run += ((double)__half2float(a) + (double)__half2float(b)) / kTapScale;
    }
    T.taps[sig].cum[2 * R + 1] = (float)run;
    auto put = [&](int op, int lane, int e, int k) {
        if (k < 0 || k > 2 * R) return;
        T.op[sig][op][0][lane][e / 2] |= (uint32_t)hi[k] << (16 * (e & 1));
        T.op[sig][op][1][lane][e / 2] |= (uint32_t)lo[k] << (16 * (e & 1));
    };
    for (int lane = 0; lane < 64; lane++)
        for (int e = 0; e < 8; e++) {
            const int gr = lane >> 4, j = lane & 15;
            for (int b = 0; b < (G::kRowOps > 1 ? 2 : 1); b++)
                for (int s = 0; s < G::kRowSteps; s++) put(G::op(b, s), lane, e, row_tap<R>(b, s, gr, j, e));
            for (int s = 0; s < G::kColOps; s++)
                if (2 * s + (e >> 2) < G::kRing) put(G::kRowOps + s, lane, e, col_tap<R>(s, gr, j, e));
        }
}

}  // namespace

void fill_strip_tables(StripTables& T) {
    std::memset(&T, 0, sizeof(T));
    fill<8>(T, SG_OPSIN);
    fill<8>(T, SG_HIGH);
    fill<8>(T, SG_MASK);
    fill<9>(T, SG_MID);
    fill<21>(T, SG_LOW);
}

int strip_height(int w0, int h0, int w1, int h1, int npairs) {
    int th = 16;
    auto wgs = [&](int t) {
        return (int64_t)npairs * ((int64_t)cdiv(w0, kStripW) * cdiv(h0, t) + (int64_t)cdiv(w1, kStripW) * cdiv(h1, t));
    };
    while (th < 128 && wgs(th) > 768) th *= 2;
    return th;
}

void launch_strip_stage(int stage, const Scales& SS, int npairs, int th, const StripTables* tab, const StripArgs& A,
                        hipStream_t st) {
    switch (stage) {
        case ST_OPSIN: launch<OpsinStage>(SS, npairs, th, tab, A, st); break;
        case ST_LOW: launch<LowStage>(SS, npairs, th, tab, A, st); break;
        case ST_MID: launch<MidStage>(SS, npairs, th, tab, A, st); break;
        default: launch<HighStage>(SS, npairs, th, tab, A, st); break;
    }
}

}  // namespace bt
}  // namespace vship
