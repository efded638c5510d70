// Device helpers shared by the Butteraugli kernels: the work planes and their
// addressing, the two-scale tile numbering, the blur factors at image edges
// and the metric's point operations.
#pragma once
#include <hip/hip_runtime.h>

#include "butter.hpp"
#include "kernel_util.hpp"

namespace vship {
namespace bt {

constexpr int kThreads = 256;
constexpr int kSigmaCount = 5;
// src/butter/gaussianblur.hpp:27-42: window max(floor(3 sigma), 8)
constexpr double kSigma[kSigmaCount] = {1.2, 1.56416327805, 2.7, 3.22489901262, 7.15593339443};
constexpr int kRad[kSigmaCount] = {8, 8, 8, 9, 21};
enum : int { SG_OPSIN = 0, SG_HIGH = 1, SG_MASK = 2, SG_MID = 3, SG_LOW = 4 };

// Work planes of one pair at one scale. Groups of three are [image][X, Y, B],
// groups of two [image][X, Y].
enum : int {
    P_LIN = 0,   // linear RGB
    P_XYB = 6,   // opsin XYB
    P_LFV = 12,  // low band, as values
    P_T = 18,    // XYB - low band
    P_MF = 24,   // middle band
    P_HFR = 30,  // high residual (before its blur)
    P_HF = 34,   // high band
    P_UHF = 38,  // ultra-high band
    P_ACS = 42,  // AC sum (all channels) without the mask term
    P_DCS = 43,  // DC sum
    P_M0 = 44,   // mask input of the reference image
    P_M1 = 45,   // mask input of the distorted image
    P_MAP = 46,  // distortion map (half scale)
    P_COUNT = 47
};

struct Scale {
    float* base;
    int w, h;
    int pitch;      // floats between rows (a multiple of 64)
    int64_t plane;  // floats between planes
    int64_t pair;   // floats between pairs
};

__device__ __forceinline__ float* plane_of(const Scale& S, int pair, int p) {
    return S.base + (int64_t)pair * S.pair + (int64_t)p * S.plane;
}

// plane_of for a pair and plane that are the same for the whole workgroup,
// held in scalar registers: without the read-first-lane the compiler folds
// the plane offset into every per-lane address as 64-bit vector arithmetic
// (the offset, not the pointer, goes through it, so that the pointer stays
// derived from the kernel argument and its loads stay global, not flat)
__device__ __forceinline__ float* plane_u(const Scale& S, int pair, int p) {
    const uint64_t v = (uint64_t)((int64_t)pair * S.pair + (int64_t)p * S.plane);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return S.base + (int64_t)(((uint64_t)hi << 32) | lo);
}

// Element off of a plane whose base is the same for the whole workgroup: a
// 32-bit byte offset from that base, which the compiler emits as the
// scalar-base + 32-bit vector-offset address form, with no 64-bit vector
// address arithmetic. Planes hold fewer than 2^30 floats (the engine checks).
__device__ __forceinline__ float& at(float* base, int off) {
    return *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + (uint64_t)((uint32_t)off * 4u));
}
__device__ __forceinline__ float at(const float* base, int off) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + (uint64_t)((uint32_t)off * 4u));
}

__host__ __device__ constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }

// Tile (x, y) of plane set z.
struct TileIdx {
    int x, y, z;
};

// Tile of workgroup b of nx * ny * nz (x fastest, then y, then z),
// XCD-aware: hardware workgroup b runs on XCD b % 8, so tiles are numbered
// such that each XCD takes one contiguous range of tile rows, and the halos
// that neighbouring tiles share are read through that XCD's L2 once.
__device__ __forceinline__ TileIdx tile_of(int b, int nx, int ny, int nz) {
    const int v = xcd_block(b, nx * ny * nz);
    // the divisions run on the vector unit; the tile is the workgroup's, so
    // it is moved to scalar registers, and the plane addresses built from it
    // stay scalar
    TileIdx t;
    t.x = __builtin_amdgcn_readfirstlane(v % nx);
    t.y = __builtin_amdgcn_readfirstlane((v / nx) % ny);
    t.z = __builtin_amdgcn_readfirstlane(v / (nx * ny));
    return t;
}

// Tile of this workgroup in a grid of one scale.
__device__ __forceinline__ TileIdx tile_of_block() {
    return tile_of(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x, gridDim.y, gridDim.z);
}

// A stage that runs both scales in one launch: the workgroups of the full
// scale come first, then those of the half scale, whose tiles fill the
// launch's tail. No stage up to the mask reads the other scale's planes. A
// launch of each scale by itself leaves most of the GPU idle where the
// picture is small (a 256 x 256 pair has 64 tiles of the blurs, 16 in the half
// scale) and pays a start and a tail of its own: 207 -> 133 us for one
// 256 x 256 pair, 477 -> 430 us for one 1920 x 1080 pair, 5.41 -> 5.34 ms for
// sixteen, all with the same results.
struct Scales {
    Scale s[2];
};

// Scale and tile of this workgroup of a two-scale launch with tiles of
// TW x TH and nz plane sets; leaves the scale in S.
template <int TW, int TH>
__device__ __forceinline__ TileIdx tile_of_scales(const Scales& SS, int nz, Scale& S) {
    const int nx0 = cdiv(SS.s[0].w, TW), ny0 = cdiv(SS.s[0].h, TH);
    const int n0 = nx0 * ny0 * nz;
    const bool half = (int)blockIdx.x >= n0;
    S = half ? SS.s[1] : SS.s[0];
    return half ? tile_of(blockIdx.x - n0, cdiv(SS.s[1].w, TW), cdiv(SS.s[1].h, TH), nz)
                : tile_of(blockIdx.x, nx0, ny0, nz);
}

// 1 / (sum of the taps inside [0, n)) at position p in [0, n) for a window of
// radius R (gaussianblur.hpp:63-65, 83-84).
template <int R, class Sums>
__device__ __forceinline__ float inv_total(const Sums* __restrict__ T, int p, int n) {
    const int lo = max(0, R - p), hi = min(2 * R, n - 1 - p + R);
    return 1.0f / (T->cum[hi + 1] - T->cum[lo]);
}

// Column and row factors of an output region [x0, x0 + OW) x [y0, y0 + OH):
// 0 outside the image.
template <int R, int OW, int OH>
__device__ __forceinline__ void edge_factors(float* colf, float* rowf, const Taps* __restrict__ T, int w, int h,
                                             int x0, int y0) {
    static_assert(OW <= 128 && OH <= 128, "factor threads");
    const int t = threadIdx.x;
    if (t < OW) {
        const int gx = x0 + t;
        colf[t] = (gx >= 0 && gx < w) ? inv_total<R>(T, gx, w) : 0.0f;
    } else if (t >= 128 && t < 128 + OH) {
        const int gy = y0 + t - 128;
        rowf[t - 128] = (gy >= 0 && gy < h) ? inv_total<R>(T, gy, h) : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// point operations (src/butter/colors.hpp, separatefrequencies.hpp:3-50,
// maskPsycho.hpp, combineMasks.hpp)
// ---------------------------------------------------------------------------
// sign(a) |a|^2.4 (colors.hpp:7-13) as 2^(2.4 log2|a|) on the hardware
// exp2/log2 units: within a few ulp of powf, which costs an order of
// magnitude more instructions. |a| is clamped to 1e-30, whose power
// underflows to exactly 0, so 0 needs no branch.
__device__ __forceinline__ float linearize(float a) {
    const float m = fmaxf(fabsf(a), 1e-30f);
    return copysignf(__builtin_amdgcn_exp2f(2.4f * __builtin_amdgcn_logf(m)), a);
}

// 19.245 ln(v + 9.971) - 23.160 with the logarithm on the hardware log2 unit
// (1 ulp; its argument is above 11) and ln 2 folded into the factor
__device__ __forceinline__ float opsin_gamma(float v) {
    constexpr float kMul = (float)(19.245013259874995 * 0.69314718055994531);
    return fmaf(kMul, __builtin_amdgcn_logf(v + 9.9710635769299145f), -23.16046239805755f);
}

__device__ __forceinline__ void opsin_absorbance(float a0, float a1, float a2, float& o0, float& o1, float& o2) {
    o0 = fmaf(0.29956550340058319f, a0, fmaf(0.63373087833825936f, a1, fmaf(0.077705617820981968f, a2, 1.7557483643287353f)));
    o1 = fmaf(0.22158691104574774f, a0, fmaf(0.69391388044116142f, a1, fmaf(0.0987313588422f, a2, 1.7557483643287353f)));
    o2 = fmaf(0.02f, a0, fmaf(0.02f, a1, fmaf(0.20480129041026129f, a2, 12.226454707163354f)));
}

// opsin response of absorbances o at a pixel whose blurred absorbances are b
// (colors.hpp:50-79); leaves the response in o
__device__ __forceinline__ void opsin_respond(float b0, float b1, float b2, float& o0, float& o1, float& o2) {
    b0 = fmaxf(fmaxf(b0, 1.7557483643287353f), 1e-4f);
    b1 = fmaxf(fmaxf(b1, 1.7557483643287353f), 1e-4f);
    b2 = fmaxf(fmaxf(b2, 12.226454707163354f), 1e-4f);
    // b >= 1.75: the hardware reciprocal (1 ulp) for the reference's division
    const float s0 = fmaxf(opsin_gamma(b0) * __builtin_amdgcn_rcpf(b0), 1e-4f);
    const float s1 = fmaxf(opsin_gamma(b1) * __builtin_amdgcn_rcpf(b1), 1e-4f);
    const float s2 = fmaxf(opsin_gamma(b2) * __builtin_amdgcn_rcpf(b2), 1e-4f);
    o0 = fmaxf(o0 * s0, 1.7557483643287353f);
    o1 = fmaxf(o1 * s1, 1.7557483643287353f);
    o2 = fmaxf(o2 * s2, 12.226454707163354f);
}

__device__ __forceinline__ float remove_range(float x, float w) { return x > w ? x - w : (x < -w ? x + w : 0.0f); }
// the reference's three cases x > w, x < -w and between as one sum with x
// clamped to [-w, w]: the same values, without branches
__device__ __forceinline__ float amplify_range(float x, float w) { return x + fminf(fmaxf(x, -w), w); }
__device__ __forceinline__ float maximum_clamp(float v, float maxval) {
    const float c = fminf(fmaxf(v, -maxval), maxval);
    return (v - c) * 0.688059627878f + c;
}

// a * b rounded to FP32 on its own: never contracted into a following add
// (where it would be kept exact), so that two values computed alike compare
// equal however they are used
__device__ __forceinline__ float mul_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

// mask input: amplitude of the high bands, compressed (maskinit + diffPrecompute)
__device__ __forceinline__ float mask_input(float hfx, float uhfx, float hfy, float uhfy) {
    // the sums of products are written as the fmas they become, so that both
    // images' are rounded alike wherever this is inlined
    const float xd = (uhfx + hfx) * 2.5f;
    const float yd = fmaf(uhfy, 0.4f, mul_rounded(hfy, 0.4f));
    // square roots of non-negative values on the hardware unit (1 ulp)
    const float m = __builtin_amdgcn_sqrtf(fmaf(xd, xd, mul_rounded(yd, yd)));
    const float mul = 6.19424080439f, bias = mul * 12.61050594197f;
    return __builtin_amdgcn_sqrtf(fmaf(mul, fabsf(m), bias)) - __builtin_amdgcn_sqrtf(bias);
}

constexpr double kMaskNorm = 1.0 / (double)(0.79079917404f * 17.83f);

__device__ __forceinline__ float mask_y(float d) {
    // hardware reciprocal (1 ulp) of a denominator above 0.8
    const float c = 2.5485944793f * __builtin_amdgcn_rcpf((0.451936922203f * d) + 0.829591754942f);
    const float r = (float)((1.0 + (double)c) * kMaskNorm);
    return r * r;
}
__device__ __forceinline__ float mask_dc_y(float d) {
    const float c = 0.505054525019f * __builtin_amdgcn_rcpf((3.87449418804f * d) + 0.20025578522f);
    const float r = (float)((1.0 + (double)c) * kMaskNorm);
    return r * r;
}

// Insert v into the three smallest values m0 <= m1 <= m2 (StoreMin3,
// maskPsycho.hpp:42-56), as a min/max network: the same three values for any
// non-NaN v as the reference's branches, which the compiler would otherwise
// lower to a private array written at a computed slot.
__device__ __forceinline__ void store_min3(float v, float& m0, float& m1, float& m2) {
    const float n2 = fminf(m2, fmaxf(m1, v));
    const float n1 = fminf(m1, fmaxf(m0, v));
    m0 = fminf(m0, v);
    m1 = n1;
    m2 = n2;
}

// One Malta term: the scaled differences of the two planes.
struct MaltaTerm {
    float n2gt, n2lt, norm1;
};

// The two weights share one hardware reciprocal (1 ulp) of
// norm1 + |a|/2 + |b|/2; the reference divides twice, and the results differ
// by rounding only.
//
// The impact term is formed without branches: with b mirrored to bm = -b when
// a < 0, the reference's two cases (maltaDiff.hpp:553-572) are the one case
// a >= 0, and too_small - bm, bm - too_big are exactly its b + too_small,
// -b - too_big (negation is exact), so the value is bit-identical.
__device__ __forceinline__ float malta_scaled_diff(float a, float b, const MaltaTerm& M) {
    const float fabs0 = fabsf(a);
    const float absval = 0.5f * fabs0 + 0.5f * fabsf(b);
    const float diff = a - b;
    const float inv = __builtin_amdgcn_rcpf(M.norm1 + absval);
    const float v = (M.n2gt * inv) * diff;
    const float scaler2 = M.n2lt * inv;
    const float too_small = 0.55f * fabs0, too_big = 1.05f * fabs0;
    const float bm = a < 0.0f ? -b : b;
    float impact = bm < too_small ? too_small - bm : (bm > too_big ? bm - too_big : 0.0f);
    impact *= scaler2;
    return diff < 0.0f ? v - impact : v + impact;
}

struct DiffParams {
    MaltaTerm malta[6];  // uhf Y, uhf X, hf Y, hf X, mf Y, mf X
    float asym_gt[2], asym_lt[2];
};

// asymmetric L2 term (simplerdiff.hpp:60-90), its cases folded as in
// malta_scaled_diff (bit-identical)
__device__ __forceinline__ float l2_asym(float a, float b, float wgt, float wlt) {
    const float diff = a - b;
    float r = wgt * diff * diff;
    const float fabs0 = fabsf(a);
    // 0.4 * |a| is a double product rounded to float in simplerdiff.hpp:69
    const float too_small = (float)(0.4 * (double)fabs0), too_big = fabs0;
    const float bm = a < 0.0f ? -b : b;
    const float v = bm < too_small ? too_small - bm : (bm > too_big ? bm - too_big : 0.0f);
    return r + wlt * v * v;
}

}  // namespace bt
}  // namespace vship
