// Butteraugli's blur stages on the matrix cores (butter_strip.hip): their
// work planes, tables and launches.
#pragma once
#include <hip/hip_runtime.h>

#include "butter_dev.hpp"

namespace vship {
namespace bt {

constexpr int kStripW = 32;           // columns of a strip
constexpr float kLinScale = 1024.0f;  // of linear RGB in the work planes these stages read
constexpr float kLinMax = 32768.0f;   // the largest magnitude there, as stored

// Work planes of the matrix-core stages, in the same arena as the general
// kernels' (the AC and DC sums, the mask inputs and the map are shared).
enum : int {
    Q_LIN = P_LIN,  // linear RGB times kLinScale, [image][R, G, B]
    Q_XY = 6,       // opsin X and Y, [image][X, Y]
    Q_DB = 10,      // difference of the images' B
    Q_T = 11,       // the same five minus their low bands
    Q_HFR = 16,     // high residual, [image][X, Y]
    Q_SD = 20,      // scaled differences of the Malta terms: ultra-high Y, X, high Y, X, middle Y, X
    Q_ACM = 26,     // L2 terms of the middle bands
    Q_COUNT = 27
};
static_assert(Q_T == Q_DB + 1 && Q_HFR == Q_T + 5 && Q_COUNT <= P_ACS, "plane layout");

// Tables of the four stages' blurs.
constexpr int kStripOps = 4;
struct StripTables {
    struct alignas(16) Blur {
        uint32_t op[kStripOps][2][64][4];  // tap operands: [h, l][lane][8 fp16]
        float cum[44];                     // sums of the taps as the operands represent them, as in Taps
    };
    Blur opsin, low, mid, high;
};
void fill_strip_tables(StripTables& T);

struct StripArgs {
    Marks* marks;
    float intensity;  // of linear RGB as stored (times kLinScale)
    DiffParams diff;
};

// Rows of a strip for npairs pairs of a w0 x h0 full and w1 x h1 half scale (a
// multiple of 16; the results do not depend on it).
int strip_height(int w0, int h0, int w1, int h1, int npairs);

// Launches stage ST_OPSIN, ST_LOW, ST_MID or ST_HIGH for both scales.
void launch_strip_stage(int stage, const Scales& SS, int npairs, int th, const StripTables* tab, const StripArgs& A,
                        hipStream_t st);

}  // namespace bt
}  // namespace vship
