// Butteraugli engine for MI355X: the two-scale distortion map and its norms
// for batches of equally sized RGB frame pairs resident in device memory
// (the metric of the reference's src/butter/main.hpp:22-195).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ssimu2_dev.hpp"  // InFmt, chroma layouts

namespace vship {
namespace bt {

// Taps of one of the five Gaussians, normalised to sum 1, and their running
// sums (cum[i] = sum of g[0..i-1]) for the renormalisation at image edges.
struct Taps {
    float g[43];
    float cum[44];
};

// One pair as the kernels read it: device planes, strides in bytes; map, if
// not null, receives the blended distortion map (row stride map_stride bytes).
// YUV formats also read bits (sample depth of the 16-bit containers), cloc
// (ChromaLoc) and the matrix's kr, kb.
struct PairDesc {
    const uint8_t* src[2][3];
    int64_t stride[2][3];
    float* map;
    int64_t map_stride;
    int32_t bits;
    int32_t cloc;
    float kr, kb;
};

// What the kernels find out about a pair. One whose values the matrix-core
// stages cannot hold is left out by every later launch of theirs, and the
// general kernels score it. The marks of the pairs follow one that says whether
// any is general: a workgroup reads that one while it works out its tile, and
// its pair's only then (read by every workgroup, the pairs' marks took the Malta
// and mask kernels 1 to 3 % longer). Sixteen 1080p pairs with a far sample each
// take 5.7 ms (the general kernels alone 5.0, 3.6 ms without such samples); with
// every stage of the strips first they took 9.1.
struct Marks {
    int32_t general;   // a value beyond the matrix-core stages
    int32_t unscaled;  // infinite linear RGB times kLinScale: the general kernels need it as it is
};

// Kernel groups, for per-kernel timing.
enum Stage : int {
    ST_INPUT = 0,  // sampling, linearisation, half-scale mean
    ST_OPSIN,      // sigma 1.2 blur + opsin dynamics
    ST_LOW,        // sigma 7.156 blur: low band, residual
    ST_MID,        // sigma 3.225 blur: middle band, X suppression
    ST_HIGH,       // sigma 1.564 blur: high / ultra-high bands
    ST_DIFF,       // Malta lines, L2 terms, mask inputs
    ST_MASK,       // sigma 2.7 blur of the masks, erosion, map, blend, norms
    ST_NORM,       // per-pair norm reduction
    ST_COUNT
};

struct StripTables;
struct Tables;

class Engine {
public:
    // Throws VshipErr (E_OutOfVRAM, E_BadDeviceArgument) on failure.
    Engine(int width, int height, int capacity, int qnorm, float intensity, int device);
    ~Engine();
    Engine(const Engine&) = delete;
    Engine& operator=(const Engine&) = delete;

    // Scores n <= capacity pairs of input format fmt (InFmt: planar RGB
    // u8/u16/f16/f32, gamma-encoded, or a limited-range YUV layout);
    // norms[3 * i .. 3 * i + 2] = Q-norm, 3-norm, max of pair i.
    // Synchronous; the work runs on stream().
    void run(int fmt, const PairDesc* pairs, int n, double* norms);

    hipStream_t stream() const { return stream_; }
    int width() const { return w_; }
    int height() const { return h_; }
    int capacity() const { return cap_; }
    int device() const { return device_; }
    int last_npairs() const { return last_n_; }

    // Per-stage times of the last submit (ms), when profiling is on.
    void set_profile(bool on) { profile_ = on; }
    bool stage_ms(float* out) const;
    // Algorithmic HBM bytes of one pair for a stage (both scales).
    uint64_t stage_bytes(int stage) const;
    // Device bytes per pair of work planes.
    static uint64_t pair_bytes(int width, int height);

private:
    // Every stage on the device: of all pairs on the matrix cores (far 0), or of
    // the far ones by the general kernels (unscaled: with the planes of linear
    // RGB made again, without their factor).
    void launch(int fmt, int pairs, int far, bool unscaled);
    void fetch_norms(int n);  // waits for them
    void release();

    int w_, h_, w2_, h2_, cap_, q_;
    float intensity_;
    int device_;
    bool profile_ = false;
    bool timed_ = false;
    int last_n_ = 0;
    int last_fmt_ = IN_RGB_F32;
    bool staged420_ = false;
    bool in_flight_ = false;
    hipStream_t stream_ = nullptr;
    float* arena_ = nullptr;
    int64_t plane0_ = 0, plane1_ = 0;
    Tables* tables_d_ = nullptr;  // owns the next two
    const Taps* taps_d_ = nullptr;
    const StripTables* strip_d_ = nullptr;
    uint8_t* block_d_ = nullptr;  // marks and descriptors of a call's pairs
    uint8_t* block_h_ = nullptr;
    double* partials_d_ = nullptr;
    double* norms_d_ = nullptr;
    double* norms_h_ = nullptr;
    int mask_tiles_ = 0;
    hipEvent_t ev_[ST_COUNT + 1] = {};
};

}  // namespace bt
}  // namespace vship
