// msceer_msc_base: what extractmsc reads out of a .grad before any
// simplification (extractmsc/extractmsc.cxx:467-556).
//
//   nodes:    one per critical cell, numbered in cell-id order
//             (MorseSmaleComplexBasic::ComputeFromGrad,
//             gi_morse_smale_complex_basic.h:676-690);
//   basins:   per vertex, the node of the minimum its V-path descends to --
//             vertex, its paired edge, the edge's other vertex, ... --
//             (FillAscendingIndexVolumeByVPaths, extractmsc.cxx:371-440,
//             written to TESTBASINS.raw);
//   mounts:   per vertex, the node of the maximum whose descending manifold
//             holds the hex at that vertex (fillGeometry of the maxima,
//             rec_man_trace_down, gi_morse_smale_complex_basic.h:1181-1198:
//             a hex paired with a facet quad belongs to the manifold of the
//             quad's other hex; TESTMOUNTS.raw), -1 where there is none.
//
// On the GPU: (1) node numbering -- every work-group counts the critical cells
// among 4096 .grad bytes, 16 a lane; one work-group scans the counts; every
// work-group then numbers its critical cells and writes, for each vertex and
// each hex, the next one on its path (itself at a critical cell, with the
// node id beside it).  (2) Every entry of the two forests follows its path
// inside a tile in LDS, then from tile to tile to its root.  (3) The labels
// from the roots' node ids.  256^3 noise: 4.0 -> 0.67 ms; jumping link by link
// with a read-back per eight links took 2.9 ms of it, the counts 0.4.  Now
// gathers across tiles (0.16 ms) and passes over memory (the rest, at 1 to 3
// TB/s) bound it.
#include <hip/hip_runtime.h>

#include "ctx.hpp"

using namespace msceer;

namespace {

constexpr int kThreads = 256;
constexpr int kPerThread = 16;
constexpr int kChunk = kThreads * kPerThread;  // cells per work-group

struct MscGeom {
    uint32_t X, Y, Z, Mx, My, Mz;
    uint64_t cells;
};

__device__ __forceinline__ bool is_critical(uint32_t b) { return ((b >> 2) & 7u) == 7u; }

// Exclusive prefix over the work-group of one value per lane; total in *total.
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* s_wave, uint32_t* total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o);
        if (lane >= (uint32_t)o) incl += t;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < kThreads / 64; w++) {
        if (w < wave) before += s_wave[w];
        all += s_wave[w];
    }
    *total = all;
    return before + incl - v;
}

// The lane's 16 cells of the chunk as dwords (cells past the end read as not
// critical): one 16-byte load where the .grad is aligned and the chunk whole.
__device__ __forceinline__ void lane_cells(const uint8_t* __restrict__ grad, uint64_t cells, uint64_t first,
                                           uint32_t w[4]) {
    if (first + kPerThread <= cells && ((uintptr_t)grad & 15u) == 0u) {
        const uint4 v = *reinterpret_cast<const uint4*>(grad + first);
        w[0] = v.x;
        w[1] = v.y;
        w[2] = v.z;
        w[3] = v.w;
        return;
    }
    for (int k = 0; k < 4; k++) {
        w[k] = 0u;
        for (int t = 0; t < 4; t++)
            if (first + 4 * k + t < cells) w[k] |= (uint32_t)grad[first + 4 * k + t] << (8 * t);
    }
}

// Bit 0 of every byte whose cell is critical (pair code 7).
__device__ __forceinline__ uint32_t critical_bytes(uint32_t w) {
    const uint32_t c = w >> 2;
    return c & (c >> 1) & (c >> 2) & 0x01010101u;
}

// Critical cells per chunk, and by dimension (coordinates only of the few that
// are critical).  Work-groups take several chunks: a group of atomics on the
// four totals per chunk took 0.4 ms at 256^3.
__global__ void __launch_bounds__(kThreads)
msc_count_kernel(const uint8_t* __restrict__ grad, MscGeom g, uint32_t chunks, uint32_t* __restrict__ chunk_counts,
                 unsigned long long* __restrict__ by_dim) {
    __shared__ uint32_t s_dim[4];
    __shared__ uint32_t s_wave[2][kThreads / 64];
    if (threadIdx.x < 4) s_dim[threadIdx.x] = 0;
    __syncthreads();
    int turn = 0;
    for (uint32_t chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x, turn ^= 1) {
        const uint64_t first = (uint64_t)chunk * kChunk + (uint64_t)threadIdx.x * kPerThread;
        uint32_t w[4];
        lane_cells(grad, g.cells, first, w);
        uint32_t n = 0;
        for (int k = 0; k < 4; k++) {
            uint32_t m = critical_bytes(w[k]);
            n += (uint32_t)__popc(m);
            for (; m; m &= m - 1) {
                const uint32_t c = (uint32_t)(first + 4 * k) + ((uint32_t)__ffs((int)m) - 1u) / 8u;
                const uint32_t q = c / g.Mx, r = q / g.My;
                atomicAdd(&s_dim[((c - q * g.Mx) & 1u) + ((q - r * g.My) & 1u) + (r & 1u)], 1u);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
        if ((threadIdx.x & 63u) == 0u) s_wave[turn][threadIdx.x >> 6] = n;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t total = 0;
            for (int k = 0; k < kThreads / 64; k++) total += s_wave[turn][k];
            chunk_counts[chunk] = total;
        }
    }
    __syncthreads();
    if (threadIdx.x < 4 && s_dim[threadIdx.x]) atomicAdd(&by_dim[threadIdx.x], (unsigned long long)s_dim[threadIdx.x]);
}

// Exclusive scan of n chunk counts in place, by one work-group, 1024 at a time.
__global__ void __launch_bounds__(1024) msc_scan_kernel(uint32_t* __restrict__ counts, uint32_t n) {
    __shared__ uint32_t s_wave[2][16];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t run = 0;
    int turn = 0;
    for (uint32_t base = 0; base < n; base += 1024u, turn ^= 1) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < n ? counts[i] : 0u;
        uint32_t incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(incl, o);
            if (lane >= (uint32_t)o) incl += t;
        }
        if (lane == 63) s_wave[turn][wave] = incl;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t k = 0; k < 16; k++) {
            if (k < wave) before += s_wave[turn][k];
            all += s_wave[turn][k];
        }
        if (i < n) counts[i] = run + before + incl - v;
        run += all;
    }
}

// Node ids of the chunk's critical cells; the next vertex / hex of every
// vertex and hex of the chunk (itself at a root, its node id or -1 in rank).
__global__ void __launch_bounds__(kThreads)
msc_link_kernel(const uint8_t* __restrict__ grad, MscGeom g, const uint32_t* __restrict__ chunk_first,
                int32_t* __restrict__ vnext, int32_t* __restrict__ vrank, int32_t* __restrict__ hnext,
                int32_t* __restrict__ hrank) {
    __shared__ uint32_t s_wave[kThreads / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kChunk;
    const uint64_t first = base + (uint64_t)threadIdx.x * kPerThread;
    uint32_t w[4], n = 0;
    lane_cells(grad, g.cells, first, w);
    for (int k = 0; k < 4; k++) n += (uint32_t)__popc(critical_bytes(w[k]));
    uint32_t total;
    uint32_t rank = chunk_first[blockIdx.x] + block_exclusive(n, s_wave, &total);
    const uint32_t Xh = g.X - 1, Yh = g.Y - 1, Zh = g.Z - 1;
    // (fewer than 2^32 cells)
    const uint32_t q0 = (uint32_t)first / g.Mx, r0 = q0 / g.My;
    uint32_t x = (uint32_t)first - q0 * g.Mx, y = q0 - r0 * g.My, z = r0;
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        if (first + k >= g.cells) continue;
        const uint32_t b = (w[k / 4] >> (8 * (k % 4))) & 255u;
        const bool crit = is_critical(b);
        const uint32_t odd = (x & 1u) + (y & 1u) + (z & 1u);
        if (odd == 0u || odd == 3u) {
            // a vertex (i, j, k) or a hex at vertex (i, j, k)
            const uint32_t i = x >> 1, j = y >> 1, kk = z >> 1;
            const bool vert = odd == 0u;
            const uint32_t nx = vert ? g.X : Xh, ny = vert ? g.Y : Yh, nz = vert ? g.Z : Zh;
            const int32_t self = (int32_t)(i + nx * (j + ny * kk));
            int32_t next = self, r = crit ? (int32_t)rank : -1;
            if (!crit) {
                // one cell along the pair direction is the paired edge / quad, two the next vertex / hex
                const uint32_t d = (b >> 2) & 7u, a = d >> 1;
                const int s = (d & 1u) ? -1 : 1;
                const int64_t ti = (int64_t)i + (a == 0 ? s : 0), tj = (int64_t)j + (a == 1 ? s : 0);
                const int64_t tk = (int64_t)kk + (a >= 2 ? s : 0);
                if (ti >= 0 && tj >= 0 && tk >= 0 && ti < nx && tj < ny && tk < nz) {
                    next = (int32_t)(ti + (int64_t)nx * (tj + (int64_t)ny * tk));
                    r = -1;
                }
                // else: off the domain (a hex paired with a boundary quad): a root of no node
            }
            (vert ? vnext : hnext)[self] = next;
            if (next == self) (vert ? vrank : hrank)[self] = r;
        }
        if (crit) rank++;
        if (++x == g.Mx) {
            x = 0;
            if (++y == g.My) {
                y = 0;
                z++;
            }
        }
    }
}

// Links followed inside a 64x4x4 tile in LDS: every entry moves on to where
// its path leaves the tile, or to its root.  (A closed path, which no gradient
// has, is left as it is; the jumps report it.)
constexpr int kTile = 1024;
constexpr uint32_t kMaxTiles = 1u << 20;  // of a launch (a grid holds fewer than 2^32 threads), from `first` on
__global__ void __launch_bounds__(kThreads)
msc_tile_kernel(int32_t* __restrict__ next, uint32_t nx, uint32_t ny, uint32_t nz, uint32_t first) {
    __shared__ uint16_t step[kTile];
    __shared__ int32_t out[kTile];
    const uint32_t tx = (nx + 63u) / 64u, ty = (ny + 3u) / 4u;
    const uint32_t tile = first + blockIdx.x;
    const uint32_t x0 = (tile % tx) * 64u, y0 = ((tile / tx) % ty) * 4u, z0 = (tile / (tx * ty)) * 4u;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const int32_t sy = (int32_t)nx, sz = (int32_t)(nx * ny);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t x = x0 + lane, y = y0 + wave, z = z0 + j, me = lane + 64u * (wave + 4u * j);
        step[me] = (uint16_t)me;
        if (x >= nx || y >= ny || z >= nz) continue;
        const int32_t self = (int32_t)(x + nx * (y + ny * z)), to = next[self];
        // one step along an axis, which a root does not take
        const int32_t d = to - self;
        out[me] = to;
        // (strides coincide where an extent is 1: the axis with room is meant)
        int32_t t = -1;
        if (d == 1 && x + 1 < nx) t = lane < 63u ? (int32_t)me + 1 : -1;
        else if (d == -1 && x > 0) t = lane > 0u ? (int32_t)me - 1 : -1;
        else if (d == sy && y + 1 < ny) t = wave < 3u ? (int32_t)me + 64 : -1;
        else if (d == -sy && y > 0) t = wave > 0u ? (int32_t)me - 64 : -1;
        else if (d == sz && z + 1 < nz) t = j < 3u ? (int32_t)me + 256 : -1;
        else if (d == -sz && z > 0) t = j > 0u ? (int32_t)me - 256 : -1;
        if (t >= 0) step[me] = (uint16_t)t;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t x = x0 + lane, y = y0 + wave, z = z0 + j, me = lane + 64u * (wave + 4u * j);
        if (x >= nx || y >= ny || z >= nz) continue;
        uint32_t t = me;
        int k = 0;
        while (step[t] != t && k < kTile) {
            t = step[t];
            k++;
        }
        if (k > 0 && k < kTile) next[x + nx * (y + ny * z)] = out[t];
    }
}

// Pointer jumping: every entry moves up to kJump links towards its root;
// *unfinished is set where it has not reached it.
constexpr int kJump = 64;
__global__ void __launch_bounds__(kThreads)
msc_jump_kernel(int32_t* __restrict__ next, uint32_t n, uint32_t* __restrict__ unfinished) {
    bool left = false;
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const int32_t p0 = next[i];
        int32_t p = p0;
        bool at_root = false;
        for (int k = 0; k < kJump; k++) {
            const int32_t q = next[p];
            at_root = q == p;
            if (at_root) break;
            p = q;
        }
        if (p != p0) next[i] = p;
        left = left || !at_root;
    }
    if (__any(left) && (threadIdx.x & 63u) == 0u) atomicOr(unfinished, 1u);
}

__global__ void __launch_bounds__(kThreads)
msc_label_kernel(MscGeom g, const int32_t* __restrict__ vnext, const int32_t* __restrict__ vrank,
                 const int32_t* __restrict__ hnext, const int32_t* __restrict__ hrank, int32_t* __restrict__ basins,
                 int32_t* __restrict__ mounts) {
    const uint64_t V = (uint64_t)g.X * g.Y * g.Z;
    for (uint64_t v = (uint64_t)blockIdx.x * kThreads + threadIdx.x; v < V; v += (uint64_t)gridDim.x * kThreads) {
        if (basins) basins[v] = vrank[vnext[v]];
        if (mounts) {
            const uint32_t i = (uint32_t)(v % g.X), j = (uint32_t)((v / g.X) % g.Y), k = (uint32_t)(v / ((uint64_t)g.X * g.Y));
            int32_t m = -1;
            if (i + 1 < g.X && j + 1 < g.Y && k + 1 < g.Z) {
                const uint32_t h = i + (g.X - 1) * (j + (g.Y - 1) * k);
                m = hrank[hnext[h]];
            }
            mounts[v] = m;
        }
    }
}

uint32_t grid_for(uint64_t n) {
    uint64_t b = (n + kThreads - 1) / kThreads;
    return (uint32_t)(b < 1 ? 1 : (b > 16384 ? 16384 : b));
}

struct Forest {
    int32_t* next;
    uint32_t nx, ny, nz;
    uint32_t n() const { return nx * ny * nz; }
};

// Jump until every entry of both forests is at its root (one read-back per
// launch of each; one launch does, unless a path crosses more than kJump tiles
// and none of its entries had moved on when it was followed).
int jump_all(msceer_ctx* ctx, const Forest* forests, int count, uint32_t* flag) {
    hipStream_t s = ctx->stream;
    for (int f = 0; f < count; f++) {
        const Forest& t = forests[f];
        if (t.n() == 0) continue;
        const uint32_t tiles = ((t.nx + 63) / 64) * ((t.ny + 3) / 4) * ((t.nz + 3) / 4);
        for (uint32_t k = 0; k < tiles; k += kMaxTiles) {
            hipLaunchKernelGGL(msc_tile_kernel, dim3(tiles - k < kMaxTiles ? tiles - k : kMaxTiles), dim3(kThreads), 0, s,
                               t.next, t.nx, t.ny, t.nz, k);
            CHECK_HIP(hipGetLastError());
        }
    }
    for (int it = 0; it < 64; it++) {
        CHECK_HIP(launch_zero(flag, 1, s));
        for (int f = 0; f < count; f++) {
            const Forest& t = forests[f];
            if (t.n() == 0) continue;
            hipLaunchKernelGGL(msc_jump_kernel, dim3(grid_for(t.n())), dim3(kThreads), 0, s, t.next, t.n(), flag);
            CHECK_HIP(hipGetLastError());
        }
        uint32_t left = 0;
        CHECK_HIP(hipMemcpyAsync(&left, flag, sizeof left, hipMemcpyDeviceToHost, s));
        CHECK_HIP(hipStreamSynchronize(s));
        if (!left) return MSCEER_OK;
    }
    return MSCEER_EHIP;  // a closed path: not a gradient
}

}  // namespace

extern "C" int msceer_msc_base(msceer_ctx* ctx, const uint8_t* grad, int64_t nx, int64_t ny, int64_t nz,
                               int32_t* basins_out, int32_t* mounts_out, int64_t* counts_out, uint32_t flags) {
    if (!ctx || !grad) return MSCEER_EINVAL;
    if (flags & ~(MSCEER_DEVICE_PTRS)) return MSCEER_EINVAL;
    int rc = check_dims(nx, ny, nz);
    if (rc) return rc;
    if (nx * ny * nz >= (int64_t)1 << 31) return MSCEER_ETOOBIG;  // int32 vertex ids and node ids
    CHECK_HIP(hipSetDevice(ctx->device));
    const Dims d = make_dims(nx, ny, nz);
    const bool dev = flags & MSCEER_DEVICE_PTRS;
    hipStream_t s = ctx->stream;
    const uint64_t V = d.verts, H = (uint64_t)(nx - 1) * (ny - 1) * (nz - 1);
    const uint32_t chunks = (uint32_t)((d.cells + kChunk - 1) / kChunk);
    // scratch: next and rank of vertices and hexes, chunk counts, dimension counts, flag
    const size_t vb = (4 * V + 255) & ~(size_t)255, hb = (4 * (H ? H : 1) + 255) & ~(size_t)255;
    const size_t cb = (4 * (size_t)chunks + 255) & ~(size_t)255;
    CHECK_HIP(ctx->scan.ensure(2 * vb + 2 * hb + cb + 256));
    uint8_t* sc = ctx->scan.as<uint8_t>();
    int32_t* vnext = reinterpret_cast<int32_t*>(sc);
    int32_t* vrank = reinterpret_cast<int32_t*>(sc + vb);
    int32_t* hnext = reinterpret_cast<int32_t*>(sc + 2 * vb);
    int32_t* hrank = reinterpret_cast<int32_t*>(sc + 2 * vb + hb);
    uint32_t* ccount = reinterpret_cast<uint32_t*>(sc + 2 * vb + 2 * hb);
    unsigned long long* by_dim = reinterpret_cast<unsigned long long*>(sc + 2 * vb + 2 * hb + cb);
    uint32_t* flag = reinterpret_cast<uint32_t*>(sc + 2 * vb + 2 * hb + cb + 64);
    const uint8_t* dgrad = grad;
    if (!dev) {
        CHECK_HIP(ctx->grad.ensure(d.cells));
        CHECK_HIP(hipMemcpyAsync(ctx->grad.ptr, grad, d.cells, hipMemcpyHostToDevice, s));
        dgrad = ctx->grad.as<uint8_t>();
    }
    int32_t* dbasins = basins_out;
    int32_t* dmounts = mounts_out;
    if (!dev && (basins_out || mounts_out)) {
        CHECK_HIP(ctx->label.ensure(8 * V));
        dbasins = basins_out ? ctx->label.as<int32_t>() : nullptr;
        dmounts = mounts_out ? ctx->label.as<int32_t>() + V : nullptr;
    }
    const MscGeom g{(uint32_t)nx, (uint32_t)ny, (uint32_t)nz, d.Mx, d.My, d.Mz, d.cells};
    CHECK_HIP(launch_zero(reinterpret_cast<uint32_t*>(by_dim), 8, s));
    hipLaunchKernelGGL(msc_count_kernel, dim3(chunks < 2048u ? chunks : 2048u), dim3(kThreads), 0, s, dgrad, g, chunks,
                       ccount, by_dim);
    CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(msc_scan_kernel, dim3(1), dim3(1024), 0, s, ccount, chunks);
    CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(msc_link_kernel, dim3(chunks), dim3(kThreads), 0, s, dgrad, g, ccount, vnext, vrank, hnext,
                       hrank);
    CHECK_HIP(hipGetLastError());
    Forest forests[2];
    int count = 0;
    if (basins_out) forests[count++] = Forest{vnext, (uint32_t)nx, (uint32_t)ny, (uint32_t)nz};
    if (mounts_out) forests[count++] = Forest{hnext, (uint32_t)nx - 1, (uint32_t)ny - 1, (uint32_t)nz - 1};
    rc = count ? jump_all(ctx, forests, count, flag) : MSCEER_OK;
    if (rc) return rc;
    if (basins_out || mounts_out) {
        hipLaunchKernelGGL(msc_label_kernel, dim3(grid_for(V)), dim3(kThreads), 0, s, g, vnext, vrank, hnext, hrank,
                           dbasins, dmounts);
        CHECK_HIP(hipGetLastError());
    }
    if (!dev) {
        if (basins_out) CHECK_HIP(hipMemcpyAsync(basins_out, dbasins, 4 * V, hipMemcpyDeviceToHost, s));
        if (mounts_out) CHECK_HIP(hipMemcpyAsync(mounts_out, dmounts, 4 * V, hipMemcpyDeviceToHost, s));
    }
    unsigned long long dims[4] = {0, 0, 0, 0};
    CHECK_HIP(hipMemcpyAsync(dims, by_dim, sizeof dims, hipMemcpyDeviceToHost, s));
    CHECK_HIP(hipStreamSynchronize(s));
    if (counts_out)
        for (int k = 0; k < 4; k++) counts_out[k] = (int64_t)dims[k];
    return MSCEER_OK;
}
