// Certain regions of the accurate labelling (GridSimplifiedExtremalRegionBuilder::
// BeginIntegration, gi_extrema_region_builder.h:806-1042) by chains and a flood.
//
// A vertex takes the label shared by all of its earlier All6 neighbours if they
// all carry one; the region seeds are labelled from the start.  Resolving the
// vertices in dependency order takes one launch per level of the DAG (880
// levels of 10 us on the 256^3 labelling volume, 9.5 ms).  The same labels
// follow without the levels:
//   chain label C(v)   the label of the seed that v's chain of earliest earlier
//                      neighbours ends at (-1: it ends at a vertex that has no
//                      earlier neighbour and is no seed)
//   bad(v)             v is no seed, and C(v) is -1 or differs from C of one of
//                      its earlier neighbours
//   v is certain, with label C(v), iff it is a seed or no bad vertex is met on
//   any way from v down through earlier neighbours (seeds end a way).
// (A certain vertex has all of its down set certain with its own label, so by
// induction C is that label all over it and nothing there is bad.  A vertex
// whose down set holds no bad vertex has C constant on it, so by induction
// every vertex of it is certain.)
// Chains are followed inside a 64x4x4 tile in LDS, then from tile to tile.
// The vertices that reach a bad one are found by a flood from the bad vertices
// along ascending edges, which needs no order: one bit per vertex, 64 vertices
// along x to a word, a work-group floods a tile of 16x16 words until nothing
// in it changes (x by doubling shifts, y and z word by word through LDS), and
// a launch floods the tiles whose rim changed in the one before.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "integrate.hpp"

namespace msceer {
namespace {

constexpr int kThreads = 256;

// Order key: value (monotone, -0 and +0 equal), then id, and the whole order
// reversed for a descending labelling.  A total order of the bits, so chains
// end even for values that have no place in the order (NaN).
__device__ __forceinline__ uint64_t order_key(float f, uint32_t id, uint64_t flip) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) == 0u) u = 0u;
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return (((uint64_t)u << 32) | id) ^ flip;
}

struct Geo {
    int X, Y, Z, words;  // words: 64-bit words per row
    int ty, tz;          // tiles of rows along y and z
};

// Planes of one bit per vertex: words along x, then y, then z.
struct Planes {
    uint64_t* up[3];  // the edge to the lower-coordinate neighbour along the axis ascends towards the vertex
    uint64_t* seed;
    uint64_t* flood;  // reaches a bad vertex
};

__device__ __forceinline__ uint64_t row_word(const Geo& g, int w, int y, int z) {
    return (uint64_t)w + (uint64_t)g.words * ((uint64_t)y + (uint64_t)g.Y * (uint64_t)z);
}

// 1. Chains and bit planes, a work-group per 64x4x4 vertices (a wave per row
// of 64): parent[v] = v where the chain ends, else the vertex where v's chain
// leaves the tile, or its end inside.
constexpr int kTX = 66, kTY = 6, kTZ = 6;
constexpr uint32_t kMaxTiles = 1u << 20;  // of a launch (a grid holds fewer than 2^32 threads), from `first` on
__global__ void __launch_bounds__(kThreads)
chain_tile_kernel(const float* __restrict__ f, Geo g, const uint8_t* __restrict__ seedmask, int32_t* __restrict__ parent,
                  Planes p, uint64_t flip, uint32_t first) {
    __shared__ float tile[kTX * kTY * kTZ];
    __shared__ uint16_t next[1024];   // in-tile successor, or itself
    __shared__ int32_t leave[1024];   // vertex the chain goes on at from there
    const uint32_t tile_id = first + blockIdx.x;
    const int w = (int)(tile_id % (uint32_t)g.words);
    const int q = (int)(tile_id / (uint32_t)g.words);
    const int nby = (g.Y + 3) / 4;
    const int x0 = w * 64, y0 = (q % nby) * 4, z0 = (q / nby) * 4;
    for (int i = threadIdx.x; i < kTX * kTY * kTZ; i += kThreads) {
        const int x = min(max(x0 - 1 + i % kTX, 0), g.X - 1);
        const int y = min(max(y0 - 1 + (i / kTX) % kTY, 0), g.Y - 1);
        const int z = min(max(z0 - 1 + i / (kTX * kTY), 0), g.Z - 1);
        tile[i] = f[(int64_t)x + (int64_t)g.X * ((int64_t)y + (int64_t)g.Y * z)];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int off[3] = {1, g.X, g.X * g.Y};
    const int toff[3] = {1, kTX, kTX * kTY};
    const int noff[3] = {1, 64, 256};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int ly = wave, lz = j;  // a wave takes one y of every z layer
        const int x = x0 + lane, y = y0 + ly, z = z0 + lz;
        const bool valid = x < g.X && y < g.Y && z < g.Z;
        const int me = lane + 64 * (ly + 4 * lz);
        const int at = (lane + 1) + kTX * ((ly + 1) + kTY * (lz + 1));
        const uint32_t v = (uint32_t)(x + g.X * (y + g.Y * z));
        const uint64_t mine = order_key(tile[at], v, flip);
        const int c[3] = {x, y, z}, n[3] = {g.X, g.Y, g.Z}, l[3] = {lane, ly, lz}, ln[3] = {64, 4, 4};
        const bool seed = valid && seedmask[v] != 0;
        uint64_t best = mine;
        int32_t to = (int32_t)v;
        int in = me;
        bool up[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const uint64_t lo = order_key(tile[at - toff[a]], v - (uint32_t)off[a], flip);
            const uint64_t hi = order_key(tile[at + toff[a]], v + (uint32_t)off[a], flip);
            const bool has_lo = c[a] > 0, has_hi = c[a] < n[a] - 1;
            up[a] = valid && has_lo && lo < mine;
            if (has_lo && lo < best) {
                best = lo;
                to = (int32_t)(v - (uint32_t)off[a]);
                in = l[a] > 0 ? me - noff[a] : -1;
            }
            if (has_hi && hi < best) {
                best = hi;
                to = (int32_t)(v + (uint32_t)off[a]);
                in = l[a] < ln[a] - 1 ? me + noff[a] : -1;
            }
        }
        if (seed || !valid) {
            to = (int32_t)v;
            in = me;
        }
        // a chain that leaves the tile here: its own successor in LDS
        next[me] = (uint16_t)(in < 0 ? me : in);
        leave[me] = to;
        const uint64_t ux = __ballot(up[0]), uy = __ballot(up[1]), uz = __ballot(up[2]), sd = __ballot(seed);
        if (lane == 0 && y < g.Y && z < g.Z) {
            const uint64_t r = row_word(g, w, y, z);
            p.up[0][r] = ux;
            p.up[1][r] = uy;
            p.up[2][r] = uz;
            p.seed[r] = sd;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int x = x0 + lane, y = y0 + wave, z = z0 + j;
        if (x >= g.X || y >= g.Y || z >= g.Z) continue;
        int t = lane + 64 * (wave + 4 * j);
        while (next[t] != t) t = next[t];
        parent[(int64_t)x + (int64_t)g.X * ((int64_t)y + (int64_t)g.Y * z)] = leave[t];
    }
}

// 2. Chain labels: every vertex but the seeds takes the label at the end of
// its chain, tile by tile.
__global__ void __launch_bounds__(kThreads)
chain_label_kernel(Geo g, const int32_t* __restrict__ parent, int32_t* label) {
    const int64_t n = (int64_t)g.X * g.Y * g.Z;
    for (int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x; v < n; v += (int64_t)gridDim.x * kThreads) {
        int32_t r = parent[v];
        if (r == (int32_t)v) continue;
        for (int32_t q = parent[r]; q != r; q = parent[r]) r = q;
        label[v] = label[r];
    }
}

// 3. Bad vertices, a wave per row word.
__global__ void __launch_bounds__(kThreads)
bad_kernel(Geo g, const int32_t* __restrict__ label, Planes p) {
    const uint64_t rows = (uint64_t)g.words * g.Y * g.Z;
    const int lane = threadIdx.x & 63;
    for (uint64_t r = (uint64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); r < rows;
         r += (uint64_t)gridDim.x * (kThreads / 64)) {
        const int w = (int)(r % (uint32_t)g.words);
        const uint32_t yz = (uint32_t)(r / (uint32_t)g.words);
        const int y = (int)(yz % (uint32_t)g.Y), z = (int)(yz / (uint32_t)g.Y);
        const int x = w * 64 + lane;
        const bool valid = x < g.X;
        const int64_t v = (int64_t)x + (int64_t)g.X * ((int64_t)y + (int64_t)g.Y * z);
        const int64_t off[3] = {1, g.X, (int64_t)g.X * g.Y};
        const uint64_t step[3] = {1, (uint64_t)g.words, (uint64_t)g.words * g.Y};
        const int c[3] = {x, y, z}, n[3] = {g.X, g.Y, g.Z};
        bool bad = false;
        if (valid && !((p.seed[r] >> lane) & 1ull)) {
            const int32_t l = label[v];
            bad = l == -1;
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if (c[a] > 0 && ((p.up[a][r] >> lane) & 1ull)) bad = bad || label[v - off[a]] != l;
                if (c[a] < n[a] - 1) {
                    // the edge to the higher-coordinate neighbour is that vertex's
                    const uint64_t word = a == 0 ? (lane < 63 ? p.up[0][r] : p.up[0][r + 1]) : p.up[a][r + step[a]];
                    const int bit = a == 0 ? (lane + 1) & 63 : lane;
                    if (!((word >> bit) & 1ull)) bad = bad || label[v + off[a]] != l;
                }
            }
        }
        const uint64_t b = __ballot(bad);
        if (lane == 0) p.flood[r] = b;
    }
}

// 4. One sweep of the flood: a work-group per tile of 16x16 row words, a lane
// per word.  dirty[tile] == sweep: a rim beside the tile changed in the sweep
// before (all tiles in the first).  A tile whose rim changes marks its
// neighbours for the next sweep; a neighbour of the same sweep may or may not
// see the change already.  Bits are only ever set, and a changed rim is read
// again by a later launch, so the flood ends complete.
__global__ void __launch_bounds__(kThreads)
flood_kernel(Geo g, Planes p, uint32_t* __restrict__ dirty, uint32_t sweep, uint32_t* __restrict__ active) {
    // active: three rotating words; this sweep reads active[sweep % 3]
    if (blockIdx.x == 0 && threadIdx.x == 0) active[(sweep + 2) % 3] = 0;
    __shared__ uint64_t rows[2][kThreads];
    // one lane decides for the work-group: a neighbour of the same sweep may be
    // writing the mark, and waves that read it apart could part ways here
    __shared__ int s_run;
    if (threadIdx.x == 0) s_run = sweep == 0 || (active[sweep % 3] != 0 && dirty[blockIdx.x] == sweep);
    __syncthreads();
    if (!s_run) return;
    const int w = (int)(blockIdx.x % (uint32_t)g.words);
    const int q = (int)(blockIdx.x / (uint32_t)g.words);
    const int ty = q % g.ty, tz = q / g.ty;
    const int t = threadIdx.x, ly = t & 15, lz = t >> 4;
    const int y = ty * 16 + ly, z = tz * 16 + lz;
    const bool row = y < g.Y && z < g.Z;
    const uint64_t r = row ? row_word(g, w, y, z) : 0;
    const uint64_t sy = (uint64_t)g.words, sz = (uint64_t)g.words * g.Y;
    const int left = g.X - w * 64;  // vertices from this word on
    const uint64_t exists = !row ? 0ull : (left >= 64 ? ~0ull : (1ull << left) - 1ull);
    const uint64_t open = row ? exists & ~p.seed[r] : 0ull;
    const bool ylo = row && y > 0, yhi = row && y < g.Y - 1, zlo = row && z > 0, zhi = row && z < g.Z - 1;
    const uint64_t upx = row ? p.up[0][r] : 0ull;
    // flow into this word's bits from its neighbours' bits
    const uint64_t from_ylo = ylo ? p.up[1][r] & open : 0ull, from_yhi = yhi ? ~p.up[1][r + sy] & open : 0ull;
    const uint64_t from_zlo = zlo ? p.up[2][r] & open : 0ull, from_zhi = zhi ? ~p.up[2][r + sz] & open : 0ull;
    const uint64_t u0 = row ? p.flood[r] : 0ull;
    uint64_t u = u0;
    // from outside the tile
    if (ly == 0 && ylo) u |= p.flood[r - sy] & from_ylo;
    if (ly == 15 && yhi) u |= p.flood[r + sy] & from_yhi;
    if (lz == 0 && zlo) u |= p.flood[r - sz] & from_zlo;
    if (lz == 15 && zhi) u |= p.flood[r + sz] & from_zhi;
    if (row && w > 0) u |= (p.flood[r - 1] >> 63) & upx & open & 1ull;
    if (row && left > 64) u |= ((p.flood[r + 1] & ~p.up[0][r + 1] & 1ull) << 63) & open;
    // along x: bit i - 1 to i where the edge ascends, i + 1 to i where it descends
    const uint64_t right = upx & open & ~1ull;
    const uint64_t leftw = ~(upx >> 1) & open & (exists >> 1);
    auto fill = [&](uint64_t b) {
        uint64_t a = b, pa = right, c = b, pc = leftw;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) {
            a |= pa & (a << k);
            pa &= pa << k;
            c |= pc & (c >> k);
            pc &= pc >> k;
        }
        return a | c;
    };
    int cur = 0;
    while (true) {
        u = fill(u);
        rows[cur][t] = u;
        __syncthreads();
        uint64_t n = u;
        if (ly > 0) n |= rows[cur][t - 1] & from_ylo;
        if (ly < 15) n |= rows[cur][t + 1] & from_yhi;
        if (lz > 0) n |= rows[cur][t - 16] & from_zlo;
        if (lz < 15) n |= rows[cur][t + 16] & from_zhi;
        const bool more = n != u;
        u = n;
        cur ^= 1;
        if (!__syncthreads_or(more ? 1 : 0)) break;
    }
    if (u == u0) return;
    p.flood[r] = u;
    const uint64_t news = u & ~u0;
    const int tiles_y = g.words, tiles_z = g.words * g.ty;
    bool marked = false;
    auto mark = [&](int tile) {
        dirty[tile] = sweep + 1;
        marked = true;
    };
    if (w > 0 && (news & 1ull)) mark((int)blockIdx.x - 1);
    if (left > 64 && (news >> 63)) mark((int)blockIdx.x + 1);
    if (ly == 0 && ty > 0) mark((int)blockIdx.x - tiles_y);
    if (ly == 15 && ty < g.ty - 1) mark((int)blockIdx.x + tiles_y);
    if (lz == 0 && tz > 0) mark((int)blockIdx.x - tiles_z);
    if (lz == 15 && tz < g.tz - 1) mark((int)blockIdx.x + tiles_z);
    if (marked) active[(sweep + 1) % 3] = 1;
}

// 5. The vertices the flood reached are not certain.
__global__ void __launch_bounds__(kThreads)
uncertain_kernel(Geo g, const uint64_t* __restrict__ flood, int32_t* __restrict__ label) {
    const uint64_t rows = (uint64_t)g.words * g.Y * g.Z;
    const int lane = threadIdx.x & 63;
    for (uint64_t r = (uint64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); r < rows;
         r += (uint64_t)gridDim.x * (kThreads / 64)) {
        const int x = (int)(r % (uint32_t)g.words) * 64 + lane;
        if (x < g.X && ((flood[r] >> lane) & 1ull)) label[(uint64_t)x + (uint64_t)g.X * (r / (uint32_t)g.words)] = -1;
    }
}

struct Layout {
    Geo g;
    uint64_t rows;
    uint32_t tiles;
    size_t dirty_off, bytes;
};

Layout layout(const VGrid& v) {
    Layout l{};
    l.g = Geo{v.X, v.Y, v.Z, (v.X + 63) / 64, (v.Y + 15) / 16, (v.Z + 15) / 16};
    l.rows = (uint64_t)l.g.words * v.Y * v.Z;
    l.tiles = (uint32_t)l.g.words * l.g.ty * l.g.tz;
    l.dirty_off = 5 * sizeof(uint64_t) * l.rows;
    l.bytes = l.dirty_off + sizeof(uint32_t) * l.tiles;
    return l;
}

Planes planes(const Layout& l, void* scratch) {
    uint64_t* p = static_cast<uint64_t*>(scratch);
    return Planes{{p, p + l.rows, p + 2 * l.rows}, p + 3 * l.rows, p + 4 * l.rows};
}

uint32_t row_blocks(uint64_t rows) { return (uint32_t)std::min<uint64_t>((rows + 3) / 4, 16384); }

}  // namespace

size_t certain_scratch_bytes(const VGrid& g) { return layout(g).bytes; }

hipError_t launch_certain_chains(const VGrid& g, const float* values, const uint8_t* seedmask, bool desc,
                                 int32_t* parent, int32_t* label, void* scratch, hipStream_t s) {
    const Layout l = layout(g);
    const Planes p = planes(l, scratch);
    const uint32_t tiles = (uint32_t)l.g.words * (uint32_t)((g.Y + 3) / 4) * (uint32_t)((g.Z + 3) / 4);
    for (uint32_t k = 0; k < tiles; k += kMaxTiles)
        hipLaunchKernelGGL(chain_tile_kernel, dim3(std::min(tiles - k, kMaxTiles)), dim3(kThreads), 0, s, values, l.g,
                           seedmask, parent, p, desc ? ~0ull : 0ull, k);
    const uint32_t blocks = (uint32_t)std::min<int64_t>((g.verts() + kThreads - 1) / kThreads, 32768);
    hipLaunchKernelGGL(chain_label_kernel, dim3(blocks), dim3(kThreads), 0, s, l.g, parent, label);
    hipLaunchKernelGGL(bad_kernel, dim3(row_blocks(l.rows)), dim3(kThreads), 0, s, l.g, label, p);
    return hipGetLastError();
}

hipError_t launch_certain_flood(const VGrid& g, void* scratch, uint32_t sweep, uint32_t* active, hipStream_t s) {
    const Layout l = layout(g);
    uint32_t* dirty = reinterpret_cast<uint32_t*>(static_cast<char*>(scratch) + l.dirty_off);
    hipLaunchKernelGGL(flood_kernel, dim3(l.tiles), dim3(kThreads), 0, s, l.g, planes(l, scratch), dirty, sweep, active);
    return hipGetLastError();
}

hipError_t launch_certain_finish(const VGrid& g, void* scratch, int32_t* label, hipStream_t s) {
    const Layout l = layout(g);
    hipLaunchKernelGGL(uncertain_kernel, dim3(row_blocks(l.rows)), dim3(kThreads), 0, s, l.g, planes(l, scratch).flood,
                       label);
    return hipGetLastError();
}

}  // namespace msceer
