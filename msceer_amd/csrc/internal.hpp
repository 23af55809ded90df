// Internal interfaces between the C ABI layer and the kernel launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace msceer {

// Vertex grid X*Y*Z and its cell complex (2X-1)(2Y-1)(2Z-1).
struct Dims {
    int X, Y, Z;
    uint32_t Mx, My, Mz;
    uint64_t cells;
    uint64_t verts;
};

inline Dims make_dims(int64_t x, int64_t y, int64_t z) {
    Dims d;
    d.X = (int)x; d.Y = (int)y; d.Z = (int)z;
    d.Mx = (uint32_t)(2 * x - 1); d.My = (uint32_t)(2 * y - 1); d.Mz = (uint32_t)(2 * z - 1);
    d.cells = (uint64_t)d.Mx * d.My * d.Mz;
    d.verts = (uint64_t)x * y * z;
    return d;
}

struct MList;

struct LstarBuffers {
    const float* values;        // device, X*Y*Z
    uint8_t* grad;              // device, cells
    const int8_t* restriction;  // device, cells, or null (steepest pass)
    const MList* list1;         // critical 1-cells: filled by every launch, read after the labelling's
    const MList* list2;         // critical 2-cells  base pass alone (extremum graphs, 1-manifolds)
    uint32_t* stats;            // device, kSubs*4: critical cells by sub-list and dimension
    uint32_t* overflow;         // device flag: a critical list ran out of room
};

// Lower-star pairing of every vertex; writes every cell byte exactly once
// with assigned/flag/pair set and ldir preset to 3 (0 for critical 3-cells).
// Lower-star kernel with brick shape `shape` (0: 64x2x2, 1: 32x4x2,
// 2: 16x4x4, 3: 8x8x4 vertices); every shape gives the same bytes.
constexpr int kLstarBricks = 4;
const char* lstar_brick_name(int shape);
hipError_t launch_lstar(const Dims& d, const LstarBuffers& b, hipStream_t s, int shape = 0);
void lstar_brick_dims(int shape, int* bx, int* by, int* bz);

// Batched launches over a group of volumes (gbatch.hpp): the unit tables,
// queues and volume table in g.
struct GBatch;
// Lower-star bricks of every volume of the group (list entries: each volume's
// cells numbered from its first[] of `items` on; restriction unused): a work-group
// per brick (blocks == 0) or `blocks` persistent work-groups claiming bricks
// (queue cleared beforehand).
hipError_t launch_lstar_batch(const GBatch& g, const LstarBuffers& b, uint32_t blocks, hipStream_t s, int shape);
// Persistent work-groups of the batched lower-star kernel one CU holds at once.
int lstar_batch_occupancy(int shape);

// ldir (ascending-manifold dimension) passes, see ldir.hip.  Geometry of the
// bit planes: the words' axis, then the other two (axis[], with the vertices
// n[] and the .grad strides cs[] along them); 64-bit words per row; flood
// tiles (16 rows each) along the rows' two axes.
struct LdirGeom {
    int axis[3];
    int n[3];
    uint32_t cs[3];
    int words, ty, tz;
};
LdirGeom ldir_geom(const Dims& d);
// Scratch: edge and quad planes, the bits reached, the tile marks, at these
// byte offsets of one device buffer of ldir_scratch_bytes().
struct LdirScratch {
    size_t rec1_off, rec2_off, bits1_off, bits2_off, dirty_off;
};
size_t ldir_scratch_bytes(const Dims& d, LdirScratch* s);
// Clears the ascending-manifold dimension bits (5-7) of n .grad bytes.
hipError_t launch_clear_ldir_bits(uint8_t* grad, int64_t n, hipStream_t st);
// Planes and start bits from the lower-star bytes; zeroes active[0..2].
hipError_t launch_ldir_planes(const Dims& d, const uint8_t* grad, void* scratch, const LdirScratch& s,
                              uint32_t* active, hipStream_t st);
// Sweep 0, 1, ... of both floods; they have ended once sweep k left
// active[(k + 1) % 3] zero (further sweeps do nothing).
hipError_t launch_ldir_flood(const Dims& d, void* scratch, const LdirScratch& s, uint32_t sweep, uint32_t* active,
                             hipStream_t st);
// Every cell's ldir from what the floods reached, if they ended within `sweeps`
// sweeps (else nothing is written).
hipError_t launch_ldir_finish(const Dims& d, uint8_t* grad, void* scratch, const LdirScratch& s, uint32_t sweeps,
                              uint32_t* active, hipStream_t st);
// Work-groups of the streaming passes of a volume, and flood tiles.
uint32_t ldir_tiles(const Dims& d);
uint32_t ldir_flood_tiles(const Dims& d);
// The same over a group of volumes, one launch each (buffers of every volume
// in its table entry; dirty: two words per flood tile of the group).
hipError_t launch_ldir_planes_group(const GBatch& b, uint32_t* active, hipStream_t st);
hipError_t launch_ldir_flood_group(const GBatch& b, uint32_t* dirty, uint32_t sweep, uint32_t* active, hipStream_t st);
hipError_t launch_ldir_finish_group(const GBatch& b, uint32_t sweeps, uint32_t* active, hipStream_t st);
// Zero n words.
hipError_t launch_zero(uint32_t* p, uint32_t n, hipStream_t s);

}  // namespace msceer
