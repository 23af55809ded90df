// Accurate 1-manifolds (lines.hip): digitized streamlines from the saddles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.hpp"

struct msceer_ctx;

namespace msceer {

struct LineStats {
    uint64_t saddles = 0;     // critical 2-cells (ASC) or 1-cells (DSC)
    uint64_t traced = 0;      // streamlines traced
    uint64_t replayed = 0;    // of those, ended before their tape by an earlier line's labels
    uint64_t voxels = 0;      // voxel traversals of all those traces
    uint64_t windows = 0;     // windows of lines traced at once
    uint64_t rounds = 0;      // evaluation rounds of all windows (enqueued)
    uint64_t cuts = 0;        // windows cut short at a line still changing after the last round
    uint64_t direct = 0;      // lines traced alone (first of a window, tape beyond the pool)
    uint64_t overflows = 0;   // windows cut short where the tape pool ran out
};

// One family of 1-manifolds: asc = from the 2-saddles up (value 4), else from
// the 1-saddles down (value 5).  grad: the steepest .grad (pairs of the
// lower-star pass); saddles (may be null: the cells are scanned): its list of
// the critical cells of that dimension, n_saddles of them; gradd: the FP64
// gradient field the streamlines follow; restr: the labels (device, one int8
// per cell) the lines are digitized into.
struct LineFamily {
    Dims d;
    const float* values;
    const uint8_t* grad;
    const MList* saddles;
    uint32_t n_saddles;
    const double4* gradd;
    int8_t* restr;
    bool asc;
    float gthr, ethr;
    int max_iters;
};

// The lines of n (at most two) families of one volume, one family after the
// other; out: n.
int run_lines(msceer_ctx* ctx, const LineFamily* families, int n, LineStats* out);

}  // namespace msceer
