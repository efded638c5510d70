// Butteraugli's blurs on the gfx950 matrix cores, fused with what surrounds
// them: opsin, low, mid and high of butter.hip's stage list, for inputs of
// ordinary range.
//
// A workgroup of four waves takes a strip of 32 columns by th rows of one pair
// and scale and streams down it in blocks of 16 rows, with all planes that the
// stage's point operations need together (both images, all channels): each
// wave blurs one plane and, where there are more than four, one 16-column half
// of another, so that the four SIMDs of a CU have the same work (a wave per
// plane, five or six, left one or two of them with twice the others': sixteen
// 1080p pairs took 0.68, 0.68 and 0.66 ms in the low, middle and opsin stages,
// with halves 0.60, 0.58 and 0.57; with streaming stores and four opsin
// workgroups per CU, see below, they take 0.56, 0.54 and 0.53, the high stage
// 0.48).
//
//   row pass     Hr(16 rows x 16 cols) = In(16 x 32 input cols) . G(32 x 16)
//   column pass  Out(16 rows x 16 cols) = G'(16 x 32 input rows) . Hr(32 x 16)
//
// on v_mfma_f32_16x16x32_f16, G being the band of taps. The input rows pass
// through a piece of LDS of the wave's own, which turns whole-row loads (16
// bytes per lane) into operands (a row per lane). The row pass leaves four rows
// of one column in a lane, which are half of its operand of the column pass as
// they stand (an operand's order in K is free, as long as the taps follow it).
// The results of all planes meet in LDS, where each thread takes two
// neighbouring pixels through the point operations.
//
// Operands are split into two fp16 parts x = h + l, both rounded to nearest,
// and all four products accumulate in FP32. A value keeps 23 significant bits of
// FP32's 24, or an absolute error of 2^-25 where its low part is subnormal: linear
// RGB is therefore stored times 2^10, and the taps carry 2^14. X and Y are
// differences and sums of values above 1.7, whose own FP32 rounding is 2^-24, so
// that 2^-25 is below what their planes hold, at any intensity. With h rounded towards
// zero and without l l, whose parts then all have their values' sign, the norms
// of 256 x 256 pairs were 0.65e-6 from their 64-bit values on average, now
// 0.40e-6 (vector kernels 0.69e-6), for 0.5 % of the time of a batch. Maps of 60
// pictures are 0.76e-6 of their mean from 64 bits on average (vector kernels
// 1.20e-6), dark ones (samples below 0.08) 2.0e-5 (4.2e-5), at an intensity of 1
// 0.92e-5 (1.84e-5), of a contrast of 0.02 3.9e-5 (6.4e-5).
// fp16 ends at 65,504, and inputs are not bounded by nature (float RGB;
// chroma far outside the gamut next to its opposite, at a high intensity):
// the input kernels check float samples against kLinMax (those of the other
// formats are below 10, of 32), and the opsin stage its results against kXybMax,
// below which no later value leaves the range (XYB minus its low band is below 2
// kXybMax, minus its middle band below 4 kXybMax = 32,768). A pair that fails,
// NaN included, is marked; the stages from there on leave it out, and the
// general kernels score it.
#include <cmath>
#include <cstring>

#include <hip/hip_fp16.h>

#include "butter_dev.hpp"
#include "butter_strip.hpp"

namespace vship {
namespace bt {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kTapScale = 16384.0f;
constexpr float kXybMax = 8192.0f;

// ---------------------------------------------------------------------------
// geometry of a strip blur of radius R
// ---------------------------------------------------------------------------
// A step takes 16 rows of kCols columns from kCol0 on (relative to the strip).
// Output block b (columns 16 b .. 16 b + 15) multiplies the 32 columns from
// 16 b on and then, if kStep2 is not 0, the next kStep2; a single block reads
// the first kCols - 16 columns from its own kCol0 on. Of the column pass the
// ring holds kRing blocks of 16 rows, the first kRowOff rows above the output
// block. LDS rows of kPitch bytes put the 16-byte operand reads of 8 or 16 lanes
// in distinct banks; at 96, without a pad, four opsin workgroups fit in a CU's
// LDS (three took 0.57 ms for sixteen 1080p pairs, four 0.54), with fewer
// conflicts than at 112.
template <int R>
struct Geo;
template <>
struct Geo<8> {  // 16 + 2 * 8 = 32 columns and rows
    static constexpr int kCol0 = -8, kCols = 48, kPitch = 96, kStep2 = 0, kRing = 2, kRowOff = 8;
};
template <>
struct Geo<9> {  // 34 columns and rows
    static constexpr int kCol0 = -12, kCols = 64, kPitch = 144, kStep2 = 16, kRing = 3, kRowOff = 16;
};
template <>
struct Geo<21> {  // 58 columns and rows
    static constexpr int kCol0 = -24, kCols = 80, kPitch = 176, kStep2 = 32, kRing = 4, kRowOff = 24;
};
template <int R>
struct Steps {
    static constexpr int kRow = Geo<R>::kStep2 ? 2 : 1, kCol = (Geo<R>::kRing + 1) / 2;
};

// Tap index of element e of lane (g, j) (g = lane / 16, j = lane % 16) in step
// s of the row pass, and of the column pass (elements 0..3 hold rows 4 g ..
// 4 g + 3 of ring block 2 s, elements 4..7 those of block 2 s + 1).
template <int R>
constexpr int row_tap(int s, int g, int j, int e) {
    const int per = s == 1 && Geo<R>::kStep2 == 16 ? 4 : 8;
    return e < per ? Geo<R>::kCol0 + 32 * s + per * g + e - j + R : -1;
}
template <int R>
constexpr int col_tap(int s, int g, int j, int e) {
    return 2 * s + (e >> 2) < Geo<R>::kRing ? -Geo<R>::kRowOff + 16 * (2 * s + (e >> 2)) + 4 * g + (e & 3) - j + R
                                            : -1;
}

// ---------------------------------------------------------------------------
// two-way fp16 split and its products
// ---------------------------------------------------------------------------
struct Op {
    u32x4 h, l;  // 8 values each
};
struct Half {
    u32x2 h, l;  // 4 values each
};

// x -> h + l, for LDS. The low parts are v_fma_mixlo/mixhi_f16 (x - h exactly,
// rounded once), written by inline assembly: the compiler makes a conversion,
// a subtraction and a conversion of each.
__device__ __forceinline__ Half split_in(const float4& x) {
    const uint32_t h0 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x.x, x.y}, f16x2));
    const uint32_t h1 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x.z, x.w}, f16x2));
    const float one = 1.0f;
    uint32_t l0, l1;
    asm("v_fma_mixlo_f16 %0, %2, %6, -%7 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %3, %6, -%7 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, %4, %6, -%8 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %1, %5, %6, -%8 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(l0), "=&v"(l1)
        : "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(one), "v"(h0), "v"(h1));
    return {u32x2{h0, h1}, u32x2{l0, l1}};
}

// half an operand: four values times s, by compiler code (they come from
// matrix instructions, whose wait states the compiler counts). The low part is
// written as the fma it is, so that every place this is inlined rounds alike:
// equal planes of the two images must give equal bands.
__device__ __forceinline__ Half split4(f32x4 v, float s) {
    Half o;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const float x = v[2 * k], y = v[2 * k + 1];
        const f16x2 h = __builtin_convertvector((f32x2){mul_rounded(x, s), mul_rounded(y, s)}, f16x2);
        const f16x2 l = __builtin_convertvector((f32x2){fmaf(x, s, -(float)h[0]), fmaf(y, s, -(float)h[1])}, f16x2);
        o.h[k] = __builtin_bit_cast(uint32_t, h);
        o.l[k] = __builtin_bit_cast(uint32_t, l);
    }
    return o;
}

__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}
// c + a . b
__device__ __forceinline__ f32x4 mma(const Op& a, const Op& b, f32x4 c) {
    c = mfma32(a.l, b.l, c);
    c = mfma32(a.l, b.h, c);
    c = mfma32(a.h, b.l, c);
    return mfma32(a.h, b.h, c);
}
// An operand of which only the first four of each lane's eight values have
// taps (the taps' other four are 0). One instruction shape throughout: with a
// 16x16x16 product accumulating onto a 16x16x32 one right before it, the results
// were wrong in two of the four accumulators under some schedules. The compiler
// (clang 22 of ROCm 7.2) puts no wait between the two, as between two products of
// one shape; whether the hardware asks for one there is not known here.
__device__ __forceinline__ Op half_op(const Half& a) {
    return {u32x4{a.h[0], a.h[1], a.h[0], a.h[1]}, u32x4{a.l[0], a.l[1], a.l[0], a.l[1]}};
}

// Orders this wave's LDS accesses before and after (its lanes exchange data
// through a region that no other wave touches).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// the stages: planes blurred together and their point operations
// ---------------------------------------------------------------------------
// remove_range without branches: the same values (of numbers)
__device__ __forceinline__ float shrink(float x, float w) { return x - fminf(fmaxf(x, -w), w); }

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
// NT: streaming stores (StripArgs)
template <bool NT>
__device__ __forceinline__ void put2(float* base, int off, const float (&v)[2]) {
    f32x2* p = reinterpret_cast<f32x2*>(&at(base, off));
    const f32x2 t = {v[0], v[1]};
    if (NT) __builtin_nontemporal_store(t, p);
    else *p = t;
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
    static constexpr int R = 8, kPlanes = 6, kSrc = Q_LIN, kCentres = 6, kWaves = 4;
    static constexpr StripTables::Blur StripTables::*kBlur = &StripTables::opsin;
    template <bool NT>
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
                ok = ok && ((y[k] <= kXybMax && o2 <= kXybMax) || (k == 1 && !X.two));
            }
            put2<NT>(plane_u(S, pair, Q_XY + 2 * im), X.g, x);
            put2<NT>(plane_u(S, pair, Q_XY + 2 * im + 1), X.g, y);
        }
        const float d[2] = {z[0][0] - z[1][0], z[0][1] - z[1][1]};
        put2<NT>(plane_u(S, pair, Q_DB), X.g, d);
        if (!ok) A.marks[0].general = A.marks[1 + pair].general = 1;
    }
};

// sigma 7.156 blur: residual XYB - low band, and the L2 terms of the low
// bands as values (separatefrequencies.hpp:142-170, 3-13; simplerdiff.hpp:38-58)
struct LowStage {
    static constexpr int R = 21, kPlanes = 5, kSrc = Q_XY, kCentres = 5, kWaves = 3;
    static constexpr StripTables::Blur StripTables::*kBlur = &StripTables::low;
    template <bool NT>
    static __device__ __forceinline__ void points(const Exchange<5>& E, const Px& X, const Centres<5>& C,
                                                  const Scale& S, int pair, const StripArgs&) {
        float lf[5][2], dc[2];
#pragma unroll
        for (int p = 0; p < 5; p++) {
            take<5>(E, p, X, lf[p]);
            const float t[2] = {C.v[p][0] - lf[p][0], C.v[p][1] - lf[p][1]};
            put2<NT>(plane_u(S, pair, Q_T + p), X.g, t);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float dx = lf[0][k] - lf[2][k], dy = lf[1][k] - lf[3][k], db = lf[4][k] + -0.362267051518f * dy;
            const float vx = dx * 33.832837186260f, vy = dy * 14.458268100570f, vb = db * 49.87984651440f;
            dc[k] = 29.2353797994f * vx * vx;
            dc[k] += 0.844626970982f * vy * vy;
            dc[k] += 0.703646627719f * vb * vb;
        }
        put2<NT>(plane_u(S, pair, P_DCS), X.g, dc);
    }
};

// sigma 3.225 blur of the residual: middle bands after their range
// operations, as Malta differences and L2 terms; high residual, X's
// suppressed by Y's (separatefrequencies.hpp:160-189)
struct MidStage {
    static constexpr int R = 9, kPlanes = 5, kSrc = Q_T, kCentres = 4, kWaves = 3;
    static constexpr StripTables::Blur StripTables::*kBlur = &StripTables::mid;
    template <bool NT>
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
                // hardware reciprocal (1 ulp) of a denominator of at least 46: the
                // general kernel divides, which gave maps and norms the same errors
                // to three digits here and took the stage 5 of 545 us longer
                hx[im][k] *= s + (yw * (1.0f - s)) * __builtin_amdgcn_rcpf(yw + yv * yv);
            }
            const float x0 = shrink(mf[0][k], 0.29f), x1 = shrink(mf[2][k], 0.29f);
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
            put2<NT>(plane_u(S, pair, Q_HFR + 2 * im), X.g, hx[im]);
            put2<NT>(plane_u(S, pair, Q_HFR + 2 * im + 1), X.g, hy[im]);
        }
        put2<NT>(plane_u(S, pair, Q_SD + 4), X.g, sy);
        put2<NT>(plane_u(S, pair, Q_SD + 5), X.g, sx);
        put2<NT>(plane_u(S, pair, Q_ACM), X.g, ac);
    }
};

// sigma 1.564 blur of the high residual: high and ultra-high bands as Malta
// differences, L2 terms and mask inputs (separatefrequencies.hpp:117-140,
// 190-200; simplerdiff.hpp:60-101; maskPsycho.hpp:24-40)
struct HighStage {
    static constexpr int R = 8, kPlanes = 4, kSrc = Q_HFR, kCentres = 4, kWaves = 4;
    static constexpr StripTables::Blur StripTables::*kBlur = &StripTables::high;
    template <bool NT>
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
                    // rounded, not contracted into the differences below: equal
                    // bands of the two images must give 0
                    uv = mul_rounded(uv, 2.69313763794f);
                    hv = mul_rounded(hv, 2.155f);
                    hv = amplify_range(hv, 0.132f);
                } else {
                    uv -= hv;
                    hv = shrink(hv, 1.5f);
                    uv = shrink(uv, 0.04f);
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
        for (int t = 0; t < 4; t++) put2<NT>(plane_u(S, pair, Q_SD + t), X.g, sd[t]);
        put2<NT>(plane_u(S, pair, P_ACS), X.g, ac);
        put2<NT>(plane_u(S, pair, P_M0), X.g, m[0]);
        put2<NT>(plane_u(S, pair, P_M1), X.g, m[1]);
    }
};

// ---------------------------------------------------------------------------
// the strip kernel
// ---------------------------------------------------------------------------
// A wave's loads of 16 rows of COLS columns, 4 columns per lane and load: whole
// rows by consecutive lanes, as many of a row as a power of two, and a last
// load of the four that are left. A load that starts in the image is read in
// place (past w up to the pitch, a multiple of 64), another at column 0 and
// masked.
template <int COLS>
struct Rows {
    static constexpr int kPer = COLS >= 64 ? 16 : 8, kMain = 16 * kPer / 64;
    static constexpr int kLoads = kMain + (COLS / 4 > kPer ? 1 : 0);
    static_assert(COLS / 4 == kPer || COLS / 4 == kPer + 4, "four loads are left of a row");
    float4 v[kLoads];
    int col[2], mask[2];  // of the main loads, of the last
    bool cols_in;
    static __device__ __forceinline__ int row(int lane, int k) {
        return k < kMain ? lane / kPer + 64 / kPer * k : lane >> 2;
    }
    static __device__ __forceinline__ int first(int lane, int k) {
        return k < kMain ? 4 * (lane % kPer) : 4 * (kPer + (lane & 3));
    }
    __device__ __forceinline__ void place(int lane, int x, int w) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int c = x + first(lane, k ? kMain : 0);
            const bool in = c >= 0 && c < w;
            col[k] = in ? c : 0;
            mask[k] = in ? (int)((1u << min(w - c, 4)) - 1u) : 0;
        }
        cols_in = x >= 0 && x + COLS <= w;
    }
    __device__ __forceinline__ void load(const float* src, int lane, int yb, int h, int pitch) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const int y = min(max(yb + row(lane, k), 0), h - 1);
            v[k] = *reinterpret_cast<const float4*>(&at(const_cast<float*>(src), y * pitch + col[k < kMain ? 0 : 1]));
        }
    }
    // the split samples into LDS rows of PITCH bytes, 0 outside the image
    template <int PITCH>
    __device__ __forceinline__ void split_to(uint8_t (*in)[16 * PITCH], int lane, int yb, int h) {
        if (!(cols_in && yb >= 0 && yb + 16 <= h)) {
#pragma unroll
            for (int k = 0; k < kLoads; k++) {
                const int y = yb + row(lane, k);
                const int m = y >= 0 && y < h ? mask[k < kMain ? 0 : 1] : 0;
                v[k].x = m & 1 ? v[k].x : 0.0f;
                v[k].y = m & 2 ? v[k].y : 0.0f;
                v[k].z = m & 4 ? v[k].z : 0.0f;
                v[k].w = m & 8 ? v[k].w : 0.0f;
            }
        }
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const Half t = split_in(v[k]);
            const int o = row(lane, k) * PITCH + 2 * first(lane, k);
            *reinterpret_cast<u32x2*>(&in[0][o]) = t.h;
            *reinterpret_cast<u32x2*>(&in[1][o]) = t.l;
        }
    }
};

template <class K, bool NT>
__global__ __launch_bounds__(kThreads, K::kWaves) void butter_strip_kernel(Scales SS, int npairs, int th,
                                                                           const StripTables* __restrict__ tab,
                                                                           StripArgs A) {
    const int any = A.marks->general;
    constexpr int R = K::R, P = K::kPlanes;
    // planes beyond the fourth: a 16-column half for each wave (two planes), or
    // for the even or the odd waves (one), in turn by workgroup
    constexpr int kExtra = P - 4, kUnits = kExtra ? 3 : 2;
    static_assert(kExtra >= 0 && kExtra <= 2, "planes of a strip");
    using G = Geo<R>;
    using N = Steps<R>;
    __shared__ Exchange<P> ex[2];
    // this step's input, of each wave its own: 16 rows of high parts, 16 of low
    __shared__ uint8_t lds[4][2][16 * G::kPitch] __attribute__((aligned(16)));
    // scale, pair and strip of this workgroup
    const int nx0 = cdiv(SS.s[0].w, kStripW), ny0 = cdiv(SS.s[0].h, th);
    const int n0 = nx0 * ny0 * npairs;
    const bool half = (int)blockIdx.x >= n0;
    const Scale S = half ? SS.s[1] : SS.s[0];
    const TileIdx ti = half ? tile_of(blockIdx.x - n0, cdiv(S.w, kStripW), cdiv(S.h, th), npairs)
                            : tile_of(blockIdx.x, nx0, ny0, npairs);
    const int pair = ti.z, x0 = ti.x * kStripW, y0 = ti.y * th;
    const int w = S.w, h = S.h, pitch = S.pitch;
    if (any && A.marks[1 + pair].general) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    auto& in = lds[wave];
    const float* src = plane_u(S, pair, K::kSrc + wave);
    const bool more = kExtra == 2 || (kExtra == 1 && ((wave ^ (blockIdx.x >> 3)) & 1) == 0);
    const int xplane = kExtra == 2 ? 4 + (wave >> 1) : 4, xblock = kExtra == 2 ? wave & 1 : wave >> 1;
    const float* xsrc = plane_u(S, pair, K::kSrc + (kExtra ? xplane : 0));

    Rows<G::kCols> V;
    Rows<G::kCols - 16> VX;
    V.place(lane, x0 + G::kCol0, w);
    V.load(src, lane, y0 - G::kRowOff, h, pitch);
    if (kExtra) {
        VX.place(lane, x0 + 16 * xblock + G::kCol0, w);
        if (more) VX.load(xsrc, lane, y0 - G::kRowOff, h, pitch);
    }

    Op rop[N::kRow], cop[N::kCol];
    const StripTables::Blur* T = &(tab->*K::kBlur);
    const u32x4* ops = reinterpret_cast<const u32x4*>(T->op);
#pragma unroll
    for (int i = 0; i < N::kRow; i++) rop[i] = {ops[2 * i * 64 + lane], ops[(2 * i + 1) * 64 + lane]};
#pragma unroll
    for (int i = 0; i < N::kCol; i++)
        cop[i] = {ops[2 * (N::kRow + i) * 64 + lane], ops[(2 * (N::kRow + i) + 1) * 64 + lane]};
    const float full = 1.0f / T->cum[2 * R + 1] * (1.0f / kTapScale);
    float kcol[kUnits];
#pragma unroll
    for (int u = 0; u < kUnits; u++) {
        const int b = u < 2 ? u : xblock;
        kcol[u] = V.cols_in ? full : inv_total<R>(T, min(x0 + 16 * b + j, w - 1), w) * (1.0f / kTapScale);
    }

    // the two pixels of this thread in the point operations
    Px X;
    X.row = threadIdx.x >> 4;
    X.col = 2 * (threadIdx.x & 15);
    const int gx = x0 + X.col;
    X.two = gx + 1 < w;

    Half ring[kUnits][G::kRing];
#pragma unroll
    for (int u = 0; u < kUnits; u++)
#pragma unroll
        for (int k = 0; k < G::kRing; k++) ring[u][k] = {u32x2{0, 0}, u32x2{0, 0}};
    // row pass of the block at byte `at0` of the staged rows into a ring
    auto row_pass = [&](int at0, Half (&rg)[G::kRing], float kc) {
        const int o = j * G::kPitch + at0 + 16 * g;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mma(Op{*reinterpret_cast<const u32x4*>(&in[0][o]), *reinterpret_cast<const u32x4*>(&in[1][o])}, rop[0],
                  acc);
        if constexpr (G::kStep2 == 32) {
            acc = mma(Op{*reinterpret_cast<const u32x4*>(&in[0][o + 64]),
                         *reinterpret_cast<const u32x4*>(&in[1][o + 64])},
                      rop[1], acc);
        } else if constexpr (G::kStep2 == 16) {
            const int o2 = j * G::kPitch + at0 + 64 + 8 * g;
            acc = mma(half_op({*reinterpret_cast<const u32x2*>(&in[0][o2]), *reinterpret_cast<const u32x2*>(&in[1][o2])}),
                      rop[1], acc);
        }
#pragma unroll
        for (int k = 0; k + 1 < G::kRing; k++) rg[k] = rg[k + 1];
        rg[G::kRing - 1] = split4(acc, kc);
    };
    auto col_pass = [&](const Half (&rg)[G::kRing]) {
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < N::kCol; s++) {
            const Half& p = rg[2 * s];
            if (2 * s + 1 < G::kRing) {
                const Half& q = rg[2 * s + 1 < G::kRing ? 2 * s + 1 : 0];
                o = mma(cop[s], Op{u32x4{p.h[0], p.h[1], q.h[0], q.h[1]}, u32x4{p.l[0], p.l[1], q.l[0], q.l[1]}}, o);
            } else {
                o = mma(cop[s], half_op(p), o);
            }
        }
        return o;
    };
    const int nout = cdiv(min(th, h - y0), 16);
    const int nblk = nout + G::kRing - 1;
#pragma unroll 1
    for (int i = 0; i < nblk; i++) {
        const int yb = y0 - G::kRowOff + 16 * i;
        const int ob = i - (G::kRing - 1), yo = y0 + 16 * ob;
        const int gy = yo + X.row;
        const bool active = ob >= 0 && gx < w && gy < h;
        X.g = gy * pitch + gx;
        wave_lds_sync();
        V.template split_to<G::kPitch>(in, lane, yb, h);
        wave_lds_sync();
        // this block's centres before the next block's loads: memory returns in
        // order, and a wait for the centres must not be one for those loads
        Centres<K::kCentres> C;
        if (active) load_centres<K::kCentres>(C, S, pair, K::kSrc, X.g);
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < nblk) V.load(src, lane, yb + 16, h, pitch);
        __builtin_amdgcn_sched_barrier(0);
        row_pass(0, ring[0], kcol[0]);
        row_pass(32, ring[1], kcol[1]);
        if (kExtra && more) {
            wave_lds_sync();
            VX.template split_to<G::kPitch>(in, lane, yb, h);
            wave_lds_sync();
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < nblk) VX.load(xsrc, lane, yb + 16, h, pitch);
            __builtin_amdgcn_sched_barrier(0);
            row_pass(0, ring[kUnits - 1], kcol[kUnits - 1]);
        }
        if (ob < 0) continue;

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
        for (int u = 0; u < kUnits; u++) {
            if (u == 2 && !more) break;
            const f32x4 o = col_pass(ring[u]);
            const int p = u < 2 ? wave : xplane, c = 16 * (u < 2 ? u : xblock) + j;
#pragma unroll
            for (int r = 0; r < 4; r++) ex[ob & 1][p][4 * g + r][c] = o[r] * krow[r];
        }
        // one barrier per block: a wave writes a buffer again only after the
        // barrier of the block between, which every reader of it has reached
        __syncthreads();
        if (active) K::template points<NT>(ex[ob & 1], X, C, S, pair, A);
    }
}

template <class K>
void launch(const Scales& SS, int n, int th, const StripTables* tab, const StripArgs& A, hipStream_t st) {
    const int64_t wgs = (int64_t)n * (cdiv(SS.s[0].w, kStripW) * cdiv(SS.s[0].h, th) +
                                      cdiv(SS.s[1].w, kStripW) * cdiv(SS.s[1].h, th));
    // Streaming stores where a stage writes more than the last-level cache
    // holds, so that the next stage would not find it there: sixteen 1080p
    // pairs 0.60 -> 0.57 ms in the low stage (0.58 -> 0.55 in the middle one, 0.57 ->
    // 0.56 in opsin, 0.50 -> 0.48 in the high one), but one pair 42 -> 47 us.
    if ((int64_t)n * (SS.s[0].plane + SS.s[1].plane) * 5 * 4 > (int64_t)256 << 20)
        butter_strip_kernel<K, true><<<dim3((unsigned)wgs), dim3(kThreads), 0, st>>>(SS, n, th, tab, A);
    else
        butter_strip_kernel<K, false><<<dim3((unsigned)wgs), dim3(kThreads), 0, st>>>(SS, n, th, tab, A);
}

template <int R>
void fill(StripTables::Blur& T, int sig) {
    double g[2 * R + 1], tot = 0.0, run = 0.0;
    uint16_t hi[2 * R + 1], lo[2 * R + 1];
    for (int k = -R; k <= R; k++) tot += g[k + R] = std::exp(-(double)k * k / (2.0 * kSigma[sig] * kSigma[sig]));
    for (int k = 0; k <= 2 * R; k++) {
        // the value the fp16 pair represents, and the sums of those values
        const float x = (float)(g[k] / tot) * kTapScale;
        const __half a = __float2half_rn(x), b = __float2half_rn(x - __half2float(a));
        hi[k] = __half_raw(a).x;
        lo[k] = __half_raw(b).x;
        T.cum[k] = (float)run;
        run += ((double)__half2float(a) + (double)__half2float(b)) / kTapScale;
    }
    T.cum[2 * R + 1] = (float)run;
    auto put = [&](int op, int lane, int e, int k) {
        if (k < 0 || k > 2 * R) return;
        T.op[op][0][lane][e / 2] |= (uint32_t)hi[k] << (16 * (e & 1));
        T.op[op][1][lane][e / 2] |= (uint32_t)lo[k] << (16 * (e & 1));
    };
    for (int lane = 0; lane < 64; lane++)
        for (int e = 0; e < 8; e++) {
            for (int s = 0; s < Steps<R>::kRow; s++) put(s, lane, e, row_tap<R>(s, lane >> 4, lane & 15, e));
            for (int s = 0; s < Steps<R>::kCol; s++)
                put(Steps<R>::kRow + s, lane, e, col_tap<R>(s, lane >> 4, lane & 15, e));
        }
}

}  // namespace

void fill_strip_tables(StripTables& T) {
    std::memset(&T, 0, sizeof(T));
    fill<OpsinStage::R>(T.opsin, SG_OPSIN);
    fill<LowStage::R>(T.low, SG_LOW);
    fill<MidStage::R>(T.mid, SG_MID);
    fill<HighStage::R>(T.high, SG_HIGH);
}

int strip_height(int w0, int h0, int w1, int h1, int npairs) {
    // About as many workgroups as are resident at once (three per CU in the low and
    // middle stages, four in the others) while the picture gives them, then taller
    // strips, whose first blocks (one to three, for the rows above) weigh less: sixteen 1080p pairs took 2.17 ms in the
    // four stages at 128 rows and 2.12 ms at 256; one 1080p pair, and a 256 x 256
    // one, the same between 512 and 1,536 workgroups.
    int th = 16;
    auto wgs = [&](int t) {
        return (int64_t)npairs * ((int64_t)cdiv(w0, kStripW) * cdiv(h0, t) + (int64_t)cdiv(w1, kStripW) * cdiv(h1, t));
    };
    while (wgs(th) > (th < 128 ? 768 : 8192) && th < 256) th *= 2;
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
