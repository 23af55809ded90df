// Ascending-manifold dimension (ldir bits) of a discrete gradient.
//
// Restates TopologicalGradientUsingAlgorithms::setAscendingManifoldDimensions
// and rec_man_trace_up_marking (gi_topological_gradient_using_algorithms.h:395-478):
// ldir = 3 everywhere; pass 1 walks from every critical 1-cell with value 2,
// pass 2 from every critical 2-cell with value 1; critical 3-cells get 0.
// Walking an item: stop if its ldir already equals the value, else set it, and
// for every cofacet t that is assigned, not critical, not paired with the item
// and whose ldir differs from the value, set ldir(t) and walk pair(t).
//
// So the marking has a closed form in terms of the items each pass reaches
// (R1: edges, R2: quads).  A critical edge is in R1; an edge paired with a
// quad t is in R1 iff another facet edge of t is; no other edge is.  R2 is the
// same one dimension up (quads paired with hexes).  Then
//   edge: 2 if in R1, else 3;
//   quad: 1 if in R2, else 2 if it is assigned, not critical and a facet edge
//         is in R1 (if its pair is a facet edge, that is in R1 iff another
//         facet is, so the pair need not be left out), else 3;
//   hex:  0 if critical, else what its pair quad would get;
//   vertex: 3.
// Reachability does not depend on the visiting order.
//
// On the GPU every edge and quad is one bit, 64 vertices along a row to a word
// (edge and quad slots belong to their lowest vertex, one of each per axis):
//  1. ldir_planes_kernel, one streaming pass over the .grad, a wave per row of
//     64 vertices: every edge's bit planes say with which of its four cofacet
//     quads it is paired, every quad's with which of its two hexes, and the
//     critical ones start R1 and R2.
//  2. ldir_flood_kernel floods R1 and R2 (both in one launch, a work-group per
//     tile of 16x16 words) until nothing changes in the tile: a word's new
//     bits are the planes' and its neighbours' words, and'ed and or'ed.  A
//     launch floods the tiles beside which something changed in the one before.
//  3. ldir_finish_kernel, one streaming pass: each vertex gets the bits of R1
//     and R2 around it, and its cells their values from those.
// What bounds it (512^3 noise): the streaming passes VALU issue (4 cycles per
// instruction of a wave) and byte accesses; between vertices in lanes and bits
// in words both change sides by a bit matrix transposition across the wave (15
// instructions for 32 words) instead of a ballot, or a mask and a select, per
// word: planes 0.68 ms (with ballots 0.81: 24 words' masks at once spill
// scalar registers), finish 1.10 ms (with masks 1.45).  Cells come by byte
// loads: as 2-byte pairs, misaligned in every other row, planes take 0.76 ms.
// The floods are bound by the updates inside a tile (LDS reads and a barrier
// per four of them, as many as the longest way in the tile) and the launches
// (as many as a way changes tiles): 2.0 ms over 24, 64^3 0.13 ms over 12.
// Walking the ways item by item (frontiers of cells over 9 bytes of records per
// vertex, visited bits by atomics) took 3.5 ms at 512^3 and 0.4 ms at 64^3,
// bound by the latency of dependent gathers, and the streaming passes around
// it, over boxes staged in LDS byte by byte, 1.17 and 1.74 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "gbatch.hpp"
#include "internal.hpp"

namespace msceer {

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kRec1 = 12;  // words of a row's edge planes: 4 per axis o, its cofacets along the other
                                // axes a1 < a2: + a1, - a1, + a2, - a2
constexpr uint32_t kRec2 = 6;   // words of a row's quad planes: +, - hex per even axis

// Bits of rows: the words run along axis 0 of the geometry's own axis order.
__device__ __forceinline__ uint32_t row_index(const LdirGeom& g, int w, int y, int z) {
    return (uint32_t)w + (uint32_t)g.words * ((uint32_t)y + (uint32_t)g.n[1] * (uint32_t)z);
}

// Buffers of one volume.
struct LdirBufs {
    uint8_t* grad;
    uint64_t* rec1;
    uint64_t* rec2;
    uint64_t* r1;  // 3 words per row: edges along axis 0, 1, 2
    uint64_t* r2;  // 3 words per row: quads with even axis 0, 1, 2
};

struct LdirArgs {
    LdirGeom g;
    LdirBufs b;
    GBatch batch;
    uint32_t* active;
    uint32_t* dirty;  // per pass and tile
    uint32_t tiles;   // flood tiles (of the group)
    uint32_t sweep;
};

// Unit of work-group i: work-groups are dealt to the XCDs round robin, so every
// XCD takes a contiguous run of the units; the pieces of a .grad line that
// neighbouring units write then meet in one L2.  A bijection of [0, n).
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t unit_of(uint32_t i, uint32_t n) {
    const uint32_t per = n / kXcds, rem = n % kXcds, xcd = i % kXcds, k = i / kXcds;
    return xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
}

// The volume of a unit of `units`, or the only one; returns the unit's index
// in its volume.
template <bool kGroup>
__device__ __forceinline__ uint32_t volume_of(LdirArgs& a, const GUnits& units, uint32_t unit, uint32_t& vol) {
    vol = 0;
    if (!kGroup) return unit;
    vol = __builtin_amdgcn_readfirstlane(unit_volume(units, unit));
    const GVol& v = a.batch.vols[vol];
    a.g = v.ldir;
    a.b = LdirBufs{v.grad, v.rec1, v.rec2, v.bits1, v.bits2};
    return unit - units.first[vol];
}

// Cells of the lane's vertices in kTileZ rows of a streaming wave: for each row
// the pairs (vertex, edge 0), (edge 1, quad 2), (edge 2, quad 1), (quad 0, hex),
// the first cell of a pair in the low byte, the one a step along axis 0
// further in the high byte; absent cells read as 0.  All loads are issued
// before any is used.
constexpr int kTileY = 4, kTileZ = 4;
struct RowCells {
    uint32_t p[4];
};
struct Stream {
    int w, y, z0, x;
    bool here, hx, hy;
    uint32_t c;  // cell of the lane's vertex in row z0
};

// Tiles of one word by 4x4 rows, a wave per y, its rows along z.
__device__ __forceinline__ Stream stream_tile(const LdirGeom& g, uint32_t tile) {
    const uint32_t ny = (uint32_t)(g.n[1] + kTileY - 1) / kTileY;
    Stream s;
    s.w = (int)(tile % (uint32_t)g.words);
    const uint32_t q = tile / (uint32_t)g.words;
    s.y = (int)(q % ny) * kTileY + (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    s.z0 = (int)(q / ny) * kTileZ;
    s.x = s.w * 64 + (int)(threadIdx.x & 63u);
    s.here = s.x < g.n[0];
    s.hx = s.x + 1 < g.n[0];
    s.hy = s.y + 1 < g.n[1];
    s.c = 2u * ((uint32_t)min(s.x, g.n[0] - 1) * g.cs[0] + (uint32_t)s.y * g.cs[1] + (uint32_t)s.z0 * g.cs[2]);
    return s;
}

__device__ __forceinline__ void load_rows(const uint8_t* __restrict__ grad, const LdirGeom& g, const Stream& s,
                                          RowCells rows[kTileZ]) {
#pragma unroll
    for (int j = 0; j < kTileZ; j++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int z = s.z0 + j;
            const bool in = z < g.n[2] && (!(k & 1) || s.hy) && (!(k & 2) || z + 1 < g.n[2]);  // the same in every lane
            const uint32_t at = s.c + (in ? 2u * g.cs[2] * (uint32_t)j + ((k & 1) ? g.cs[1] : 0u) + ((k & 2) ? g.cs[2] : 0u)
                                          : 0u);
            const uint32_t v = (uint32_t)grad[at] | (s.hx ? (uint32_t)grad[at + g.cs[0]] << 8 : 0u);
            rows[j].p[k] = in && s.here ? v : 0u;
        }
}

// Pair code of an assigned cell, 8 of any other.
__device__ __forceinline__ uint32_t code_of(uint32_t b) { return (b & 1u) ? (b >> 2) & 7u : 8u; }

// Bit matrix transposition in each half of the wave: bit c of lane l goes to
// bit l of lane c.
struct Transpose {
    uint32_t turn[5], keep[5];  // step i exchanges with lane ^ (1 << i)
    __device__ explicit Transpose(uint32_t lane) {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const uint32_t m = i == 0 ? 0x55555555u : i == 1 ? 0x33333333u : i == 2 ? 0x0F0F0F0Fu : i == 3 ? 0x00FF00FFu
                                                                                                         : 0x0000FFFFu;
            const bool up = (lane >> i) & 1u;
            turn[i] = up ? 1u << i : 32u - (1u << i);
            keep[i] = up ? ~m : m;
        }
    }
    __device__ __forceinline__ uint32_t step(uint32_t v, uint32_t other, int i) const {
        return (keep[i] & v) | (~keep[i] & __builtin_amdgcn_alignbit(other, other, turn[i]));
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t v) const {
        v = step(v, (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 16 << 10 | 31), 4);       // lane ^ 16
        v = step(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 15, 15, true), 3);    // lane ^ 8: half a row on
        v = step(v, (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 4 << 10 | 31), 2);        // lane ^ 4
        v = step(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 15, 15, true), 1);     // lane ^ 2: quad 2 3 0 1
        return step(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 15, 15, true), 0);  // lane ^ 1: quad 1 0 3 2
    }
};

template <bool kGroup>
__global__ void __launch_bounds__(kThreads) ldir_planes_kernel(LdirArgs a) {
    if (blockIdx.x == 0 && threadIdx.x < 3) a.active[threadIdx.x] = 0u;
    uint32_t vol;
    const uint32_t tile = volume_of<kGroup>(a, a.batch.tiles, unit_of(blockIdx.x, gridDim.x), vol);
    const LdirGeom& g = a.g;
    const Stream s = stream_tile(g, tile);
    if (s.y >= g.n[1]) return;
    const uint32_t lane = threadIdx.x & 63u;
    RowCells rows[kTileZ];
    load_rows(a.b.grad, g, s, rows);
    // after the transposition lane 8 * k + code of each half holds which of the
    // half's vertices have edge (quad) k paired by that code: the half word the
    // lane stores, if it is one
    const int k = (int)(lane >> 3) & 3, code = (int)(lane & 7u);
    const int along = code >> 1;  // axis of the code
    const int h = along == g.axis[0] ? 0 : (along == g.axis[1] ? 1 : 2);
    uint64_t *e = nullptr, *q = nullptr;
    if (k < 3 && code == 7) {
        e = a.b.r1 + k;
        q = a.b.r2 + k;
    } else if (k < 3 && code < 6) {
        if (h != k) e = a.b.rec1 + (4 * k + 2 * (h - (h > k ? 1 : 0)) + (code & 1));
        if (h == k) q = a.b.rec2 + (2 * k + (code & 1));
    }
    const uint32_t pe = code == 7 ? 3u : kRec1, pq = code == 7 ? 3u : kRec2;
    const Transpose transpose(lane);
    auto hot = [](uint32_t b) { return (b & 1u) << ((b >> 2) & 7u); };
#pragma unroll
    for (int j = 0; j < kTileZ; j++) {
        const int z = s.z0 + j;
        if (z >= g.n[2]) break;
        const uint32_t* p = rows[j].p;
        const uint32_t te = transpose(hot(p[0] >> 8) | hot(p[1]) << 8 | hot(p[2]) << 16);
        const uint32_t tq = transpose(hot(p[3]) | hot(p[2] >> 8) << 8 | hot(p[1] >> 8) << 16);
        const uint64_t row = row_index(g, s.w, s.y, z);
        if (e) reinterpret_cast<uint32_t*>(e + pe * row)[lane >> 5] = te;
        if (q) reinterpret_cast<uint32_t*>(q + pq * row)[lane >> 5] = tq;
    }
}

// ---- floods ------------------------------------------------------------------

constexpr int kRim = 18;  // 16 rows and one more on each side

struct Words3 {
    uint64_t w[3];
};

__device__ __forceinline__ uint64_t load_lds(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void store_lds(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// One update of a row's words from its own and its neighbours' (at(k, dy, dz):
// word k of the row dy, dz further on), m: the row's planes.  "x + 1" of a word
// is its bits shifted right, "x - 1" left.
template <class At>
__device__ __forceinline__ Words3 edges_update(const Words3& r, const uint64_t m[12], At at) {
    auto xp = [](uint64_t v) { return v >> 1; };
    auto xm = [](uint64_t v) { return v << 1; };
    const uint64_t r0 = r.w[0], r1 = r.w[1], r2 = r.w[2];
    const uint64_t a0 = at(0, 1, 0), a2 = at(2, 1, 0);                      // y + 1
    const uint64_t b0 = at(0, -1, 0), b1 = at(1, -1, 0), b2 = at(2, -1, 0);  // y - 1
    const uint64_t c0 = at(0, 0, 1), c1 = at(1, 0, 1);                      // z + 1
    const uint64_t e0 = at(0, 0, -1), e1 = at(1, 0, -1), e2 = at(2, 0, -1);  // z - 1
    const uint64_t f2 = at(2, 1, -1), h1 = at(1, -1, 1);                    // y + 1, z - 1; y - 1, z + 1
    Words3 n = r;
    // an edge along o paired with the quad towards +a: the edge along o at + a,
    // the edges along a at the vertex and at + o; towards -a: the same from - a
    n.w[0] |= (m[0] & (a0 | r1 | xp(r1))) | (m[1] & (b0 | b1 | xp(b1))) | (m[2] & (c0 | r2 | xp(r2))) |
              (m[3] & (e0 | e2 | xp(e2)));
    n.w[1] |= (m[4] & (xp(r1) | r0 | a0)) | (m[5] & (xm(r1) | xm(r0) | xm(a0))) | (m[6] & (c1 | r2 | a2)) |
              (m[7] & (e1 | e2 | f2));
    n.w[2] |= (m[8] & (xp(r2) | r0 | c0)) | (m[9] & (xm(r2) | xm(r0) | xm(c0))) | (m[10] & (a2 | r1 | c1)) |
              (m[11] & (b2 | b1 | h1));
    return n;
}
template <class At>
__device__ __forceinline__ Words3 quads_update(const Words3& r, const uint64_t m[6], At at) {
    auto xp = [](uint64_t v) { return v >> 1; };
    auto xm = [](uint64_t v) { return v << 1; };
    const uint64_t r0 = r.w[0], r1 = r.w[1], r2 = r.w[2];
    const uint64_t a1 = at(1, 1, 0), c2 = at(2, 0, 1);                      // y + 1; z + 1
    const uint64_t b0 = at(0, -1, 0), b1 = at(1, -1, 0), b2 = at(2, -1, 0), h2 = at(2, -1, 1);
    const uint64_t e0 = at(0, 0, -1), e1 = at(1, 0, -1), e2 = at(2, 0, -1), f1 = at(1, 1, -1);
    Words3 n = r;
    // a quad paired with the hex at the vertex: the hex's five other facets (two
    // per axis, at the vertex and one further on); with the hex one back: the
    // same from there
    n.w[0] |= (m[0] & (xp(r0) | r1 | a1 | r2 | c2)) | (m[1] & xm(r0 | r1 | a1 | r2 | c2));
    n.w[1] |= (m[2] & (a1 | r0 | xp(r0) | r2 | c2)) | (m[3] & (b1 | b0 | xp(b0) | b2 | h2));
    n.w[2] |= (m[4] & (c2 | r0 | xp(r0) | r1 | a1)) | (m[5] & (e2 | e0 | xp(e0) | e1 | f1));
    return n;
}

// dirty[tile of a pass] == sweep: something beside the tile changed in the
// sweep before (all tiles run in the first).  A tile that changed marks the
// tiles that read the changed rows for the next sweep; a neighbour of the same
// sweep may or may not see the change already.  Bits are only ever set, and a
// change is read again by a later launch, so the floods end complete.
// active: three rotating words; this sweep reads active[sweep % 3].
constexpr int kInner = 4;  // updates between two barriers (512^3, 64^3: 2.01 ms, 0.14 ms; of 2: 2.01, 0.145; of 8: 2.09, 0.14)
template <bool kGroup>
__global__ void __launch_bounds__(kThreads) ldir_flood_kernel(LdirArgs a) {
    if (blockIdx.x == 0 && threadIdx.x == 0) a.active[(a.sweep + 2) % 3] = 0u;
    const uint32_t sweep = a.sweep;
    const int pass = blockIdx.x >= a.tiles ? 1 : 0;
    const uint32_t unit = unit_of(blockIdx.x - (pass ? a.tiles : 0u), a.tiles);
    __shared__ uint64_t lds[3][kRim][kRim];
    // one lane decides for the work-group: a neighbour of the same sweep may be
    // writing the mark, and waves that read it apart could part ways here
    __shared__ int s_run;
    if (threadIdx.x == 0)
        s_run = sweep == 0 || (a.active[sweep % 3] != 0u && a.dirty[unit + (pass ? a.tiles : 0u)] == sweep);
    __syncthreads();
    if (!s_run) return;
    uint32_t vol;
    const uint32_t tile = volume_of<kGroup>(a, a.batch.floods, unit, vol);
    const LdirGeom& g = a.g;
    uint64_t* const bits = pass ? a.b.r2 : a.b.r1;
    const int w = (int)(tile % (uint32_t)g.words);
    const uint32_t q = tile / (uint32_t)g.words;
    const int ty = (int)(q % (uint32_t)g.ty), tz = (int)(q / (uint32_t)g.ty);
    const int t = (int)threadIdx.x, ly = t & 15, lz = t >> 4;
    const int y = ty * 16 + ly, z = tz * 16 + lz;
    const bool row = y < g.n[1] && z < g.n[2];
    const uint32_t r = row ? row_index(g, w, y, z) : 0u;
    const int32_t sy = g.words, sz = g.words * g.n[1];
    // the tile's words and those of the rows around it
    for (int i = t; i < kRim * kRim; i += kThreads) {
        const int iy = i % kRim, iz = i / kRim;
        const int gy = ty * 16 + iy - 1, gz = tz * 16 + iz - 1;
        const bool in = gy >= 0 && gz >= 0 && gy < g.n[1] && gz < g.n[2];
        const uint64_t* p = bits + 3ull * (in ? row_index(g, w, gy, gz) : 0u);
#pragma unroll
        for (int k = 0; k < 3; k++) lds[k][iz][iy] = in ? p[k] : 0ull;
    }
    uint64_t m[kRec1];
#pragma unroll
    for (uint32_t k = 0; k < kRec1; k++)
        m[k] = !row ? 0ull : (pass == 0 ? a.b.rec1[(uint64_t)kRec1 * r + k]
                                        : (k < kRec2 ? a.b.rec2[(uint64_t)kRec2 * r + k] : 0ull));
    Words3 u{};
    if (row)
#pragma unroll
        for (int k = 0; k < 3; k++) u.w[k] = bits[3ull * r + k];
    const Words3 old = u;
    // bits that come across the word's ends: bit 63 from the next word's first
    // vertex, bit 0 from the last one of the word before
    if (row) {
        auto word = [&](int k, int dw, int dy, int dz) -> uint64_t {
            if (y + dy < 0 || y + dy >= g.n[1] || z + dz < 0 || z + dz >= g.n[2]) return 0ull;
            return bits[3ll * ((int64_t)r + dw + (int64_t)sy * dy + (int64_t)sz * dz) + k];
        };
        if (w + 1 < g.words) {
            auto first = [&](int k, int dy, int dz) { return word(k, 1, dy, dz) << 63; };
            if (pass == 0) {
                const uint64_t n1 = first(1, 0, 0), n2 = first(2, 0, 0);
                u.w[0] |= (m[0] & n1) | (m[1] & first(1, -1, 0)) | (m[2] & n2) | (m[3] & first(2, 0, -1));
                u.w[1] |= m[4] & n1;
                u.w[2] |= m[8] & n2;
            } else {
                const uint64_t n0 = first(0, 0, 0);
                u.w[0] |= m[0] & n0;
                u.w[1] |= (m[2] & n0) | (m[3] & first(0, -1, 0));
                u.w[2] |= (m[4] & n0) | (m[5] & first(0, 0, -1));
            }
        }
        if (w > 0) {
            auto last = [&](int k, int dy, int dz) { return word(k, -1, dy, dz) >> 63; };
            if (pass == 0) {
                const uint64_t p0 = last(0, 0, 0);
                u.w[1] |= m[5] & (last(1, 0, 0) | p0 | last(0, 1, 0));
                u.w[2] |= m[9] & (last(2, 0, 0) | p0 | last(0, 0, 1));
            } else {
                u.w[0] |= m[1] & (last(0, 0, 0) | last(1, 0, 0) | last(1, 1, 0) | last(2, 0, 0) | last(2, 0, 1));
            }
        }
    }
    __syncthreads();
    if (row)
#pragma unroll
        for (int k = 0; k < 3; k++) store_lds(&lds[k][lz + 1][ly + 1], u.w[k]);
    __syncthreads();
    auto at = [&](int k, int dy, int dz) { return load_lds(&lds[k][lz + 1 + dz][ly + 1 + dy]); };
    // rounds until one changes nothing: the words in LDS are then those every
    // lane computed with
    while (true) {
        bool more = false;
#pragma unroll 1
        for (int j = 0; j < kInner; j++) {
            const Words3 n = pass == 0 ? edges_update(u, m, at) : quads_update(u, m, at);
            bool ch = false;
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (n.w[k] != u.w[k]) {
                    store_lds(&lds[k][lz + 1][ly + 1], n.w[k]);
                    ch = true;
                }
            u = n;
            more = more || ch;
        }
        if (!__syncthreads_or(more ? 1 : 0)) break;
    }
    uint64_t news = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (u.w[k] != old.w[k]) bits[3ull * r + k] = u.w[k];
        news |= u.w[k] & ~old.w[k];
    }
    if (!news) return;
    // the tiles that read this row: beside it along y and z, along both where
    // one is ahead and the other behind, and in the next and the previous word
    uint32_t* const dirty = a.dirty + (pass ? a.tiles : 0u);
    bool marked = false;
    auto mark = [&](int dw, int dy, int dz) {
        if (ty + dy < 0 || ty + dy >= g.ty || tz + dz < 0 || tz + dz >= g.tz) return;
        dirty[(int64_t)unit + dw + (int64_t)g.words * (dy + (int64_t)g.ty * dz)] = sweep + 1;
        marked = true;
    };
    const bool ylo = ly == 0, yhi = ly == 15, zlo = lz == 0, zhi = lz == 15;
    if (ylo) mark(0, -1, 0);
    if (yhi) mark(0, 1, 0);
    if (zlo) mark(0, 0, -1);
    if (zhi) mark(0, 0, 1);
    if (yhi && zlo) mark(0, 1, -1);
    if (ylo && zhi) mark(0, -1, 1);
    if ((news & 1ull) && w > 0) {  // read by the word before: from its rows here, at y + 1 and at z + 1
        mark(-1, 0, 0);
        if (yhi) mark(-1, 1, 0);
        if (zhi) mark(-1, 0, 1);
    }
    if ((news >> 63) && w + 1 < g.words) {  // by the next word: from its rows here, at y - 1 and at z - 1
        mark(1, 0, 0);
        if (ylo) mark(1, -1, 0);
        if (zlo) mark(1, 0, -1);
    }
    if (marked) a.active[(sweep + 1) % 3] = 1u;
}

// ---- the ldir bits -------------------------------------------------------------

// Words a row of the finish needs, one per lane of each half wave: in the order
// of the bits that a vertex has after the transposition.  The first five are
// also needed at the vertex one further along axis 0; the last five hold that
// vertex where it is in the next word.
enum FinishBit : uint32_t {
    kE1, kE2, kE2y, kE1z, kQ0, kE0, kE0y, kE0z, kE0yz, kQ1, kQ2, kQ1y, kQ2z, kNext, kFinishWords = kNext + 5,
    kFurther = 20  // where a lane puts the five of the next vertex
};
// array (0: r1, 1: r2) << 5 | word << 3 | next word << 2 | y + 1 << 1 | z + 1
__constant__ uint8_t kFinishAt[kFinishWords] = {0x08, 0x10, 0x12, 0x09, 0x20, 0x00, 0x02, 0x01, 0x03,
                                                0x28, 0x30, 0x2a, 0x31, 0x0c, 0x14, 0x16, 0x0d, 0x24};

template <bool kGroup>
__global__ void __launch_bounds__(kThreads) ldir_finish_kernel(LdirArgs a) {
    // the floods are not done after `sweep` sweeps: another finish follows
    if (a.active[a.sweep % 3] != 0u) return;
    uint32_t vol;
    const uint32_t tile = volume_of<kGroup>(a, a.batch.tiles, unit_of(blockIdx.x, gridDim.x), vol);
    const LdirGeom& g = a.g;
    const Stream s = stream_tile(g, tile);
    const uint32_t lane = threadIdx.x & 63u;
    uint8_t* __restrict__ const grad = a.b.grad;
    if (s.y < g.n[1]) {
        const uint32_t d0 = 2u * (uint32_t)g.axis[0], d1 = 2u * (uint32_t)g.axis[1], d2 = 2u * (uint32_t)g.axis[2];
        RowCells rows[kTileZ];
        load_rows(grad, g, s, rows);
        // the lane's half word of every row
        const uint32_t slot = lane & 31u, sel = slot < kFinishWords ? kFinishAt[slot] : 0u;
        const int dw = (sel >> 2) & 1, dy = (sel >> 1) & 1, dz = sel & 1;
        const bool in = slot < kFinishWords && s.w + dw < g.words && s.y + dy < g.n[1];
        const uint32_t* const src = reinterpret_cast<const uint32_t*>(((sel & 32u) ? a.b.r2 : a.b.r1) + ((sel >> 3) & 3u)) +
                                    (lane >> 5);
        uint32_t words[kTileZ];
#pragma unroll
        for (int j = 0; j < kTileZ; j++) {
            const int z = s.z0 + j;
            const bool ok = in && z + dz < g.n[2];
            const uint32_t v = src[6ull * (ok ? row_index(g, s.w + dw, s.y + dy, z + dz) : row_index(g, s.w, s.y, s.z0))];
            words[j] = ok ? v : 0u;
        }
        const Transpose transpose(lane);
#pragma unroll
        for (int j = 0; j < kTileZ; j++) {
            const int z = s.z0 + j;
            if (z >= g.n[2]) break;
            const bool hz = z + 1 < g.n[2];
            uint32_t t = transpose(words[j]);
            const uint32_t after = (uint32_t)__builtin_amdgcn_readfirstlane((int)t) >> kNext;
            uint32_t n = (uint32_t)__builtin_amdgcn_mov_dpp((int)t, 0x130, 15, 15, true);  // of lane + 1
            n = lane == 63u ? after : n;
            t = (t & ((1u << kNext) - 1u)) | n << kFurther;
            auto any = [&](uint32_t m) { return (t & m) != 0u; };
            auto bit = [](uint32_t k) { return 1u << k; };
            auto on = [](uint32_t k) { return 1u << (kFurther + k); };  // one further along axis 0
            // quads with a facet edge in R1, at the row and where a hex's other facets lie
            const bool m0 = any(bit(kE1) | bit(kE2) | bit(kE2y) | bit(kE1z));
            const bool m1 = any(bit(kE2) | on(kE2) | bit(kE0) | bit(kE0z));
            const bool m2 = any(bit(kE1) | on(kE1) | bit(kE0) | bit(kE0y));
            const bool m0x = any(on(kE1) | on(kE2) | on(kE2y) | on(kE1z));
            const bool m1y = any(bit(kE2y) | on(kE2y) | bit(kE0y) | bit(kE0yz));
            const bool m2z = any(bit(kE1z) | on(kE1z) | bit(kE0z) | bit(kE0yz));
            auto value = [&](uint32_t in_r2, bool m) { return any(in_r2) ? 1u : (m ? 2u : 3u); };
            const uint32_t v0 = value(bit(kQ0), m0), v1 = value(bit(kQ1), m1), v2 = value(bit(kQ2), m2);
            // a hex gets what its pair quad would: the vertex's own quads, or those one further on
            const uint32_t of_code = v0 << (2 * d0 + 2) | value(on(kQ0), m0x) << 2 * d0 | v1 << (2 * d1 + 2) |
                                     value(bit(kQ1y), m1y) << 2 * d1 | v2 << (2 * d2 + 2) |
                                     value(bit(kQ2z), m2z) << 2 * d2;
            const uint32_t* p = rows[j].p;
            auto edge = [&](uint32_t k) { return any(bit(k)) ? 2u : 3u; };
            // (a quad that is critical or unassigned gets no 2)
            auto quad = [&](uint32_t b, uint32_t v) { return v == 2u && code_of(b) >= 7u ? 3u : v; };
            const uint32_t hc = code_of(p[3] >> 8);
            auto with = [](uint32_t two, uint32_t lo, uint32_t hi) { return (two & 0x1F1Fu) | lo << 5 | hi << 13; };
            const uint32_t out[4] = {
                with(p[0], (p[0] >> 5) & 7u, edge(kE0)),  // (the vertex keeps its 3)
                with(p[1], edge(kE1), quad(p[1] >> 8, v2)), with(p[2], edge(kE2), quad(p[2] >> 8, v1)),
                with(p[3], quad(p[3], v0), hc == 7u ? (p[3] >> 13) & 7u : (hc < 7u ? (of_code >> 2u * hc) & 3u : 3u))};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (((k & 1) && !s.hy) || ((k & 2) && !hz)) continue;  // the same in every lane
                uint8_t* const at = grad + (s.c + 2u * g.cs[2] * (uint32_t)j + ((k & 1) ? g.cs[1] : 0u) +
                                            ((k & 2) ? g.cs[2] : 0u));
                if (g.cs[0] == 1u && s.hx) {
                    const uint16_t two = (uint16_t)out[k];
                    __builtin_memcpy(at, &two, 2);
                } else if (s.here) {
                    at[0] = (uint8_t)out[k];
                    if (s.hx) at[g.cs[0]] = (uint8_t)(out[k] >> 8);
                }
            }
        }
    }
    if (kGroup && a.batch.times) {
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(&a.batch.times[2 * vol + 1], batch_clock());
    }
}

__global__ void zero_kernel(uint32_t* p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

uint64_t rows_of(const LdirGeom& g) { return (uint64_t)g.words * g.n[1] * g.n[2]; }

LdirArgs one_volume(const Dims& d, const uint8_t* grad, void* scratch, const LdirScratch& s) {
    uint8_t* base = static_cast<uint8_t*>(scratch);
    LdirArgs a{};
    a.g = ldir_geom(d);
    a.b.grad = const_cast<uint8_t*>(grad);
    a.b.rec1 = reinterpret_cast<uint64_t*>(base + s.rec1_off);
    a.b.rec2 = reinterpret_cast<uint64_t*>(base + s.rec2_off);
    a.b.r1 = reinterpret_cast<uint64_t*>(base + s.bits1_off);
    a.b.r2 = reinterpret_cast<uint64_t*>(base + s.bits2_off);
    a.dirty = reinterpret_cast<uint32_t*>(base + s.dirty_off);
    a.tiles = ldir_flood_tiles(d);
    return a;
}

}  // namespace

// Words run along x, or along the longest axis where x is short: a row of
// fewer than 32 vertices would leave most of its words empty.
LdirGeom ldir_geom(const Dims& d) {
    const int n[3] = {d.X, d.Y, d.Z};
    const uint32_t cs[3] = {1u, d.Mx, d.Mx * d.My};
    int first = 0;
    if (n[0] < 32)
        for (int k = 1; k < 3; k++)
            if (n[k] > n[first]) first = k;
    LdirGeom g{};
    g.axis[0] = first;
    g.axis[1] = first == 1 ? 0 : 1;
    g.axis[2] = first == 2 ? 0 : 2;
    for (int k = 0; k < 3; k++) {
        g.n[k] = n[g.axis[k]];
        g.cs[k] = cs[g.axis[k]];
    }
    g.words = (g.n[0] + 63) / 64;
    g.ty = (g.n[1] + 15) / 16;
    g.tz = (g.n[2] + 15) / 16;
    return g;
}

size_t ldir_scratch_bytes(const Dims& d, LdirScratch* s) {
    const uint64_t rows = rows_of(ldir_geom(d));
    auto al = [](size_t n) { return (n + 255) & ~(size_t)255; };
    const size_t r1 = al(8 * kRec1 * rows), r2 = al(8 * kRec2 * rows), b = al(8 * 3 * rows);
    const size_t dirty = al(2 * sizeof(uint32_t) * (size_t)ldir_flood_tiles(d));
    if (s) {
        s->rec1_off = 0;
        s->rec2_off = r1;
        s->bits1_off = r1 + r2;
        s->bits2_off = r1 + r2 + b;
        s->dirty_off = r1 + r2 + 2 * b;
    }
    return r1 + r2 + 2 * b + dirty;
}

uint32_t ldir_tiles(const Dims& d) {
    const LdirGeom g = ldir_geom(d);
    return (uint32_t)g.words * (uint32_t)((g.n[1] + kTileY - 1) / kTileY) *
           (uint32_t)((g.n[2] + kTileZ - 1) / kTileZ);
}

uint32_t ldir_flood_tiles(const Dims& d) {
    const LdirGeom g = ldir_geom(d);
    return (uint32_t)g.words * (uint32_t)g.ty * (uint32_t)g.tz;
}

__global__ void __launch_bounds__(256) clear_ldir_words_kernel(uint32_t* __restrict__ w, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) w[i] &= 0x1F1F1F1Fu;
}

__global__ void __launch_bounds__(256) clear_ldir_bytes_kernel(uint8_t* __restrict__ g, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) g[i] &= 0x1Fu;
}

hipError_t launch_clear_ldir_bits(uint8_t* grad, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    // 4-byte words where the buffer is aligned, bytes for the rest
    const int64_t lead = (int64_t)((4 - (reinterpret_cast<uintptr_t>(grad) & 3)) & 3);
    const int64_t head = lead < n ? lead : n;
    const int64_t words = (n - head) / 4;
    const int64_t tail = n - head - 4 * words;
    auto blocks = [](int64_t m) { return (unsigned)std::min<int64_t>((m + 255) / 256, 8192); };
    if (head) hipLaunchKernelGGL(clear_ldir_bytes_kernel, dim3(1), dim3(256), 0, st, grad, head);
    if (words)
        hipLaunchKernelGGL(clear_ldir_words_kernel, dim3(blocks(words)), dim3(256), 0, st,
                           reinterpret_cast<uint32_t*>(grad + head), words);
    if (tail) hipLaunchKernelGGL(clear_ldir_bytes_kernel, dim3(1), dim3(256), 0, st, grad + head + 4 * words, tail);
    return hipGetLastError();
}

hipError_t launch_ldir_planes(const Dims& d, const uint8_t* grad, void* scratch, const LdirScratch& s,
                              uint32_t* active, hipStream_t st) {
    LdirArgs a = one_volume(d, grad, scratch, s);
    a.active = active;
    hipLaunchKernelGGL(ldir_planes_kernel<false>, dim3(ldir_tiles(d)), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ldir_flood(const Dims& d, void* scratch, const LdirScratch& s, uint32_t sweep, uint32_t* active,
                             hipStream_t st) {
    LdirArgs a = one_volume(d, nullptr, scratch, s);
    a.active = active;
    a.sweep = sweep;
    hipLaunchKernelGGL(ldir_flood_kernel<false>, dim3(2 * a.tiles), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ldir_finish(const Dims& d, uint8_t* grad, void* scratch, const LdirScratch& s, uint32_t sweeps,
                              uint32_t* active, hipStream_t st) {
    LdirArgs a = one_volume(d, grad, scratch, s);
    a.active = active;
    a.sweep = sweeps;
    hipLaunchKernelGGL(ldir_finish_kernel<false>, dim3(ldir_tiles(d)), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ldir_planes_group(const GBatch& b, uint32_t* active, hipStream_t st) {
    LdirArgs a{};
    a.batch = b;
    a.active = active;
    hipLaunchKernelGGL(ldir_planes_kernel<true>, dim3(b.tiles.total), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ldir_flood_group(const GBatch& b, uint32_t* dirty, uint32_t sweep, uint32_t* active, hipStream_t st) {
    LdirArgs a{};
    a.batch = b;
    a.active = active;
    a.dirty = dirty;
    a.tiles = b.floods.total;
    a.sweep = sweep;
    hipLaunchKernelGGL(ldir_flood_kernel<true>, dim3(2 * b.floods.total), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ldir_finish_group(const GBatch& b, uint32_t sweeps, uint32_t* active, hipStream_t st) {
    LdirArgs a{};
    a.batch = b;
    a.active = active;
    a.sweep = sweeps;
    hipLaunchKernelGGL(ldir_finish_kernel<true>, dim3(b.tiles.total), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_zero(uint32_t* p, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint32_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(zero_kernel, dim3(blocks), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

}  // namespace msceer
