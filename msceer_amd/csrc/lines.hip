// Accurate 1-manifolds: streamlines from the saddles, digitized into the
// restriction labels of the conforming gradient.
//
// Semantics restated (reference file:line):
//   driver:     ondemandaccurate.cxx:254-500 (ReIntegrateUpFrom2Saddles,
//               ReIntegrateDownFrom1Saddles), 1075-1091
//   streamline: gi_numeric_streamline_integrator.h:734-788 (ASC), 1018-1072 (DSC)
//   digitizing: gi_numeric_streamline_integrator.h:566-700 (ASC), 824-985 (DSC)
//   checkers:   gi_advection_checker.h:59-100 (TerminateNearAssignedHex / Vert)
//   advection:  gi_adaptive_euler_advector.h:51-305 (sign +1 ASC, -1 DSC)
//
// ASC: the critical 2-cells (quads) of the steepest gradient, in decreasing
// (value of the highest vertex, cell id) order; DSC: the critical 1-cells
// (edges), in increasing value, decreasing id.  Each saddle's seeds are the
// cells a short V-path search reaches (hexes ASC, vertices DSC, at most six);
// from each seed, in order, one FP64 streamline (uphill ASC, downhill DSC)
// labels the cells it crosses -- for each crossed face, the cell it leaves and
// the face -- with the target value (4 ASC, 5 DSC), stops as soon as it steps
// into a cell (the voxel ASC, the nearest vertex DSC) that already carries the
// target, or near the boundary; after its streamlines the saddle itself takes
// the target.  One reference thread runs this in order, so later streamlines
// stop on earlier ones: the result is defined by that order.
//
// On the GPU the order is kept exactly, over windows of streamlines ("lines";
// the saddle's own label is a line without a trace):
//  1. every line of the window is traced at once, one lane a line, and records
//     a tape: what it would ask of the labels if only its own stopped it
//     (lines_core.hpp).  Nothing is read from the labels but, in later
//     windows, the committed ones;
//  2. rounds: every line is evaluated along its tape, one wave a line, against
//     the labels the lines gave in the round before (per cell the lowest line
//     that gives it; an earlier line's label counts, a later one's does not).
//     Line k of the window is exact once the lines before it are, so round k
//     at the latest; in practice the rounds stop changing anything after five
//     to ten, and then every line is exact;
//  3. the labels are committed; the next window follows.
// A line whose tape does not fit the pool ends its window; first in a window,
// it is traced alone, in order.  The windows after one that ended early are
// shorter, and grow again while their tapes leave room.
//
// What bounds it: the tracing, the latency of the longest streamline's steps
// (FP64 chains of a few hundred cycles and, at each voxel entered, a gather
// of 8 corners): 2.7 ms a family on the 256^3 labelling volume.  A tape holds
// 20 to 40 entries on average, so a round is a few dependent reads per line
// (90 us).  Tracing interacting lines again in order, a lane per component,
// took 77 ms there and reading labels at every step of the first trace 42 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <hipcub/hipcub.hpp>

#include "ctx.hpp"
#include "integrate.hpp"
#include "lines.hpp"
#include "lines_core.hpp"

#pragma clang fp contract(off)

namespace msceer {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ uint32_t wave_append(bool want, uint32_t* counter) {
    const uint64_t m = __ballot(want);
    if (!m) return 0;
    const int lane = (int)(threadIdx.x & 63u);
    const int leader = __ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    return base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
}

// ---- the saddles and their seeds -------------------------------------------

// Key of saddle c: the float key of the value of its highest vertex (by value,
// id) -- negated for DSC -- << 32 | cell id.
__device__ __forceinline__ uint64_t saddle_key(const CellGeom& m, int X, int Y, const float* __restrict__ f, int asc,
                                               uint32_t c) {
    int64_t x, y, z;
    m.xyz(c, x, y, z);
    int64_t best = -1;
    for (int k = 0; k < 8; k++) {
        if (((k & 1) && !(x & 1)) || ((k & 2) && !(y & 1)) || ((k & 4) && !(z & 1))) continue;
        const int64_t vx = (x >> 1) + (k & 1), vy = (y >> 1) + ((k >> 1) & 1), vz = (z >> 1) + (k >> 2);
        const int64_t v = vx + (int64_t)X * (vy + (int64_t)Y * vz);
        if (best < 0 || f[v] > f[best] || (!(f[best] > f[v]) && v > best)) best = v;
    }
    const float val = f[best];
    return ((uint64_t)value_key(asc ? val : -1.0f * val) << 32) | (uint64_t)c;
}

// Keys of the critical cells of dimension sdim: sorted descending, this is the
// reference's processing order (pairs (value, id) sorted ascending and taken
// from the end).
__global__ void __launch_bounds__(kThreads)
line_saddles_kernel(const uint8_t* __restrict__ grad, CellGeom m, int X, int Y, const float* __restrict__ f,
                    int sdim, int asc, uint64_t* __restrict__ keys, uint32_t* count, uint32_t cap) {
    const uint64_t C = (uint64_t)m.sxy * (uint64_t)m.Mz;
    const uint64_t stride = (uint64_t)gridDim.x * kThreads;
    for (uint64_t base = (uint64_t)blockIdx.x * kThreads; base < C; base += stride) {
        const uint64_t c = base + threadIdx.x;
        bool want = false;
        if (c < C && critical(grad, (uint32_t)c)) {
            int64_t x, y, z;
            m.xyz((uint32_t)c, x, y, z);
            want = (int)((x & 1) + (y & 1) + (z & 1)) == sdim;
        }
        const uint32_t at = wave_append(want, count);
        if (want && at < cap) keys[at] = saddle_key(m, X, Y, f, asc, (uint32_t)c);
    }
}

// The same keys from the lower-star pass's list of the critical cells of that
// dimension (in any order).
__global__ void __launch_bounds__(kThreads)
line_saddle_list_kernel(MList list, CellGeom m, int X, int Y, const float* __restrict__ f, int asc,
                        uint64_t* __restrict__ keys, uint32_t n) {
    __shared__ uint32_t prefix[kSubs + 2];
    const uint32_t total = min(mlist_prefix(list, prefix), n);
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads) {
        const uint32_t c = mlist_at(list, prefix, i);
        keys[i] = saddle_key(m, X, Y, f, asc, c);
    }
}

// Per saddle (rank k in processing order): its seeds in slots 7k .. 7k+5 and
// the saddle in slot 7k+6.
__global__ void __launch_bounds__(kThreads)
line_seeds_kernel(const uint8_t* __restrict__ grad, CellGeom m, const uint64_t* __restrict__ keys, uint32_t n,
                  int asc, uint32_t* __restrict__ slots) {
    const uint32_t k = blockIdx.x * kThreads + threadIdx.x;
    if (k < n) saddle_seeds(grad, m, (uint32_t)keys[k], asc != 0, slots + 7 * (uint64_t)k);
}

struct LineArgs {
    GradSrc<double> src;
    VGrid g;
    CellGeom m;
    const uint32_t* slots;  // 7 per saddle
    int8_t* restr;
    int8_t target;
    bool asc;
    double gthr, ethr;
    int max_iters;
    TapePool pool;
    uint64_t* wmask;   // per chunk: list entries whose cell carries the target after them
    uint32_t* active;  // lines of the window with a tape
    uint32_t* head;    // their first chunks
    uint32_t* ended;   // where they ended: slots along the tape, 0 at its end
    uint32_t* stamp[2];  // per cell: round tag << kLineBits | lowest line of the window giving it its label
    uint32_t* ctl;     // kLcWords words
};

enum LineCtl : int {
    kLcOverflow = 0,  // lowest line whose tape did not fit the pool
    kLcActive = 1,    // lines of the window with a tape
    kLcTraced = 2,    // streamlines traced
    kLcVoxels = 3,    // voxel traversals
    kLcTop = 4,       // next free chunk of the pool
    kLcCut = 5,       // streamlines that ended before their tape
    kLcChanged = 6,   // three words: lines a round changed (rotating)
    kLcLowest = 9,    // three words: the lowest of them
    kLcWords = 12
};

// Stamps: the tag falls from round to round, so that a round's stamps replace
// older ones under atomicMin and nothing is cleared between rounds, windows or
// calls; the arrays are refilled when the tags run out.
constexpr int kLineBits = 20;
constexpr uint32_t kLineMask = (1u << kLineBits) - 1u;
constexpr uint32_t kTopTag = (1u << (32 - kLineBits)) - 2u;  // the first tag after a refill
constexpr uint32_t kMaxRounds = 512;                         // of one window

// 1. Tapes of lines [w0, w1): a lane per line, a wave per work-group, so that
// the longest lines' waves share no work-group's registers and LDS.
constexpr int kTapeThreads = 64;
__global__ void __launch_bounds__(kTapeThreads) line_tape_kernel(LineArgs a, uint32_t w0, uint32_t w1) {
    __shared__ uint32_t hist[kHistory * kTapeThreads];
    const uint32_t i = w0 + blockIdx.x * kTapeThreads + threadIdx.x;
    const uint32_t c = i < w1 && i % 7 != 6 ? a.slots[i] : kNoLine;
    uint32_t first = kNoLine;
    if (c != kNoLine) {
        TapeLabels lab{a.restr, a.target, w0 > 0, a.pool, hist + threadIdx.x, (uint32_t)kTapeThreads};
        lab.geom = a.m;
        uint32_t vox = 0;
        trace_line(a.src, a.g, a.m, c, a.asc, a.gthr, a.ethr, a.max_iters, lab, &vox);
        lab.finish();
        if (lab.over) atomicMin(&a.ctl[kLcOverflow], i);
        else first = lab.head;
        atomicAdd(&a.ctl[kLcTraced], 1u);
        atomicAdd(&a.ctl[kLcVoxels], vox);
    }
    const uint32_t at = wave_append(first != kNoLine, &a.ctl[kLcActive]);
    if (first != kNoLine) {
        a.active[at] = i;
        a.head[at] = first;
        a.ended[at] = 0;
    }
}

// The lines of a window end before the first one whose tape did not fit.
__device__ __forceinline__ uint32_t window_end(const LineArgs& a, uint32_t w1) { return min(a.ctl[kLcOverflow], w1); }

// Links of a tape: for every entry the line's previous kList entry of the same
// cell.  A wave per line; pairs of chunks whose cells' boxes do not meet are
// skipped, so a long tape costs little more than its length.
struct CellBox {
    int lo[3], hi[3];
};
__global__ void __launch_bounds__(kTapeThreads) line_links_kernel(LineArgs a) {
    __shared__ uint32_t s_chunk[kMaxTapeChunks];
    __shared__ CellBox s_box[kMaxTapeChunks];
    const uint32_t lane = threadIdx.x;
    const uint32_t n_active = a.ctl[kLcActive];
    for (uint32_t t = blockIdx.x; t < n_active; t += gridDim.x) {
        uint32_t q = 0;
        for (uint32_t ch = a.head[t]; ch != kNoLine; q++) {
            uint64_t* const e = a.pool.slots + (uint64_t)ch * kTapeChunk;
            const uint64_t mine = e[lane];
            const uint32_t next = __builtin_amdgcn_readfirstlane((uint32_t)mine);
            const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(mine >> 32));
            const bool valid = lane >= 1 && lane <= n;
            const uint32_t c = (uint32_t)mine, hi = (uint32_t)(mine >> 32);
            const bool list = valid && ((hi >> kKindShift) & 3u) == kList;
            int64_t p[3] = {0, 0, 0};
            if (valid) a.m.xyz(c, p[0], p[1], p[2]);
            CellBox box;
            for (int d = 0; d < 3; d++) {
                int lo = valid ? (int)p[d] : 0x7fffffff, hi3 = valid ? (int)p[d] : -1;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    lo = min(lo, __shfl_xor(lo, o));
                    hi3 = max(hi3, __shfl_xor(hi3, o));
                }
                box.lo[d] = lo;
                box.hi[d] = hi3;
            }
            uint32_t prev = kNoPrev;
            for (uint32_t b = 0; b < q; b++) {
                const CellBox& o = s_box[b];
                bool meet = true;
                for (int d = 0; d < 3; d++) meet = meet && o.lo[d] <= box.hi[d] && box.lo[d] <= o.hi[d];
                if (!meet) continue;
                const uint32_t och = s_chunk[b];
                const uint64_t theirs = a.pool.slots[(uint64_t)och * kTapeChunk + lane];
                const uint32_t on = kTapeChunk - 1;  // every chunk but the last is full
                const uint32_t ohi = (uint32_t)(theirs >> 32);
                const uint64_t olist = __ballot(lane >= 1 && lane <= on && ((ohi >> kKindShift) & 3u) == kList);
                for (uint64_t rest = olist; rest; rest &= rest - 1) {
                    const int j = __ffsll((unsigned long long)rest) - 1;
                    if (__shfl((uint32_t)theirs, j) == c) prev = och * kTapeChunk + (uint32_t)j;
                }
            }
            const uint64_t lists = __ballot(list);
            for (uint64_t rest = lists; rest; rest &= rest - 1) {
                const int j = __ffsll((unsigned long long)rest) - 1;
                if (__shfl(c, j) == c && (uint32_t)j < lane) prev = ch * kTapeChunk + (uint32_t)j;
            }
            if (valid && prev != kNoPrev) e[lane] = (uint64_t)((hi & ~kNoPrev) | prev) << 32 | c;
            if (lane == 0) {
                s_chunk[q] = ch;
                s_box[q] = box;
            }
            __syncthreads();
            ch = next;
        }
        __syncthreads();
    }
}

// The k-th slot of a saddle's own label from line w0 on.
__device__ __forceinline__ uint64_t saddle_slot(uint32_t w0, uint32_t k) {
    return (uint64_t)w0 + (6u - w0 % 7u) + 7ull * k;
}

// 2. One round: every line of [w0, wc) evaluated along its tape against the
// stamps of the round before (tag + 1), its labels stamped with `tag`.  A
// round after one that changed nothing has nothing to do.
__global__ void __launch_bounds__(kThreads)
line_round_kernel(LineArgs a, uint32_t w0, uint32_t w1, uint32_t round, uint32_t tag) {
    const uint32_t wc = window_end(a, w1);
    uint32_t* const changed = a.ctl + kLcChanged;
    uint32_t* const lowest = a.ctl + kLcLowest;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        changed[(round + 1) % 3] = 0;
        lowest[(round + 1) % 3] = kNoLine;
    }
    if (round > 0 && changed[(round + 2) % 3] == 0) return;
    const uint32_t* const in = a.stamp[round & 1];
    uint32_t* const out = a.stamp[(round & 1) ^ 1];
    // the saddles' own labels
    const uint64_t threads = (uint64_t)gridDim.x * kThreads;
    for (uint64_t i = saddle_slot(w0, blockIdx.x * kThreads + threadIdx.x); i < wc; i += 7 * threads)
        atomicMin(&out[a.slots[i]], tag << kLineBits | (uint32_t)(i - w0));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * (kThreads / 64);
    const uint32_t n_active = a.ctl[kLcActive];
    uint32_t n_changed = 0, low = kNoLine;
    for (uint32_t t = blockIdx.x * (kThreads / 64) + threadIdx.x / 64; t < n_active; t += waves) {
        const uint32_t line = __builtin_amdgcn_readfirstlane(a.active[t]);
        if (line >= wc) continue;
        TapeState s;
        uint32_t ended = 0, ord = 0;
        bool diff = false;
        for (uint32_t ch = a.head[t]; ch != kNoLine && !ended; ord++) {
            const uint64_t e = a.pool.slots[(uint64_t)ch * kTapeChunk + lane];
            const uint32_t next = __builtin_amdgcn_readfirstlane((uint32_t)e);
            const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(e >> 32));
            const bool valid = lane >= 1 && lane <= n;
            const uint32_t c = (uint32_t)e, hi = (uint32_t)(e >> 32), kind = (hi >> kKindShift) & 3u;
            bool labelled = false;
            if (valid) {
                const uint32_t v = in[c];
                labelled = round > 0 && (v >> kLineBits) == tag + 1 && (v & kLineMask) < line - w0;
                if (w0 > 0) labelled = labelled || a.restr[c] == a.target;
            }
            const uint64_t before = a.wmask[ch];
            auto own = [&](uint32_t k, uint64_t w) {
                const uint32_t p = __builtin_amdgcn_readlane(hi, k) & kNoPrev;
                uint64_t word = w;
                if (p / kTapeChunk != ch)
                    word = __hip_atomic_load(&a.wmask[p / kTapeChunk], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return ((word >> (p % kTapeChunk)) & 1ull) != 0;
            };
            uint32_t at = 0;
            const uint64_t w = tape_chunk(s, n, __ballot(valid && kind <= kExit), __ballot(valid && kind == kExit),
                                          __ballot(valid && kind == kStop), __ballot(valid && (hi & kFirst)),
                                          __ballot(labelled), __ballot(valid && (hi & kNoPrev) != kNoPrev), own, &at);
            if (before != w) {
                diff = true;
                if (lane == 0)
                    __hip_atomic_store(&a.wmask[ch], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if ((w >> lane) & 1ull) atomicMin(&out[c], tag << kLineBits | (line - w0));
            if (at) ended = ord * kTapeChunk + at;
            ch = next;
        }
        if (round == 0 || diff || a.ended[t] != ended) {
            n_changed++;
            low = line < low ? line : low;
            if (lane == 0) a.ended[t] = ended;
        }
    }
    if (lane == 0 && n_changed) {
        atomicAdd(&changed[round % 3], n_changed);
        atomicMin(&lowest[round % 3], low);
    }
}

// 3. Commit the labels of the lines before `end`, unless round `last` still
// changed some (check).
__global__ void __launch_bounds__(kThreads)
line_commit_kernel(LineArgs a, uint32_t w0, uint32_t end, uint32_t last, bool check) {
    if (check && a.ctl[kLcChanged + last % 3] != 0) return;
    const uint32_t cut = window_end(a, end);
    const uint64_t threads = (uint64_t)gridDim.x * kThreads;
    for (uint64_t i = saddle_slot(w0, blockIdx.x * kThreads + threadIdx.x); i < cut; i += 7 * threads)
        a.restr[a.slots[i]] = a.target;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * (kThreads / 64);
    const uint32_t n_active = a.ctl[kLcActive];
    uint32_t n_cut = 0;
    for (uint32_t t = blockIdx.x * (kThreads / 64) + threadIdx.x / 64; t < n_active; t += waves) {
        const uint32_t line = __builtin_amdgcn_readfirstlane(a.active[t]);
        if (line >= cut) continue;
        const uint32_t ended = a.ended[t];
        uint32_t ord = 0;
        for (uint32_t ch = a.head[t]; ch != kNoLine && !(ended && ord * kTapeChunk >= ended); ord++) {
            const uint64_t e = a.pool.slots[(uint64_t)ch * kTapeChunk + lane];
            const uint64_t w = a.wmask[ch];
            if ((w >> lane) & 1ull) a.restr[(uint32_t)e] = a.target;
            ch = __builtin_amdgcn_readfirstlane((uint32_t)e);
        }
        n_cut += ended ? 1u : 0u;
    }
    if (lane == 0 && n_cut) atomicAdd(&a.ctl[kLcCut], n_cut);
}

// A line traced alone, in order (first of its window, its tape beyond the pool).
__global__ void line_direct_kernel(LineArgs a, uint32_t i) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    DirectLabels lab{a.restr, a.target};
    const uint32_t c = a.slots[i];
    if (c == kNoLine) return;
    if (i % 7 == 6) {
        lab.write(c);
        return;
    }
    uint32_t vox = 0;
    trace_line(a.src, a.g, a.m, c, a.asc, a.gthr, a.ethr, a.max_iters, lab, &vox);
    a.ctl[kLcTraced] += 1;
    a.ctl[kLcVoxels] += vox;
}

__global__ void line_ctl_init_kernel(uint32_t* ctl, bool all) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        ctl[kLcOverflow] = kNoLine;
        ctl[kLcActive] = 0;
        ctl[kLcTop] = 0;
        for (int k = 0; k < 3; k++) {
            ctl[kLcChanged + k] = 0;
            ctl[kLcLowest + k] = kNoLine;
        }
        if (all) {
            ctl[kLcTraced] = 0;
            ctl[kLcVoxels] = 0;
            ctl[kLcCut] = 0;
        }
    }
}

__global__ void __launch_bounds__(kThreads) line_fill_kernel(uint32_t* p, uint64_t n, uint32_t v) {
    const uint64_t stride = (uint64_t)gridDim.x * kThreads;
    for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) p[i] = v;
}

inline uint32_t blocks_for(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, (n + kThreads - 1) / kThreads); }

}  // namespace

// Window of lines traced at once (bounds the tapes' scratch; line numbers in
// the stamps have kLineBits bits).  The
// environment variable MSCEER_LINE_WINDOW (8 .. 2^20) sets a smaller one,
// which tests use to exercise many windows on small volumes; as
// MSCEER_LINE_CHUNKS (1 .. 2^22) does for the pool's chunks and
// MSCEER_LINE_ROUNDS (2 .. 512) for the rounds of a window.
constexpr uint32_t kWindow = 1u << kLineBits;
constexpr uint32_t kMaxChunks = 1u << 22;

static uint32_t env_size(const char* name, uint32_t least, uint32_t most, uint32_t otherwise) {
    if (const char* e = getenv(name)) {
        const long v = atol(e);
        if (v >= (long)least && v <= (long)most) return (uint32_t)v;
    }
    return otherwise;
}

uint32_t line_window() { return env_size("MSCEER_LINE_WINDOW", 8, kWindow, kWindow); }

namespace {

// A family's lines: their seeds and scratch, the first window's tapes enqueued.
struct LineJob {
    uint64_t nslots = 0;
    uint32_t W = 0;
    LineArgs a{};
};

// Lines [w0, w1): tapes and links.
int enqueue_tapes(const LineArgs& a, uint32_t w0, uint32_t w1, hipStream_t s) {
    const uint32_t n = w1 - w0;
    hipLaunchKernelGGL(line_ctl_init_kernel, dim3(1), dim3(64), 0, s, a.ctl, false);
    hipLaunchKernelGGL(line_tape_kernel, dim3((n + kTapeThreads - 1) / kTapeThreads), dim3(kTapeThreads), 0, s, a, w0, w1);
    hipLaunchKernelGGL(line_links_kernel, dim3(std::min<uint32_t>(n, 8192)), dim3(kTapeThreads), 0, s, a);
    CHECK_HIP(hipGetLastError());
    return MSCEER_OK;
}

// Number of lines' saddles: of the list, else counted by a scan over the cells.
int count_saddles(msceer_ctx* ctx, const LineFamily& f, const CellGeom& m, uint32_t* S) {
    *S = f.n_saddles;
    if (f.saddles) return MSCEER_OK;
    hipStream_t s = ctx->stream;
    CHECK_HIP(launch_zero(ctl_dev(ctx) + kCtlCount, 1, s));
    hipLaunchKernelGGL(line_saddles_kernel, dim3(2048), dim3(kThreads), 0, s, f.grad, m, f.d.X, f.d.Y, f.values,
                       f.asc ? 2 : 1, f.asc ? 1 : 0, nullptr, ctl_dev(ctx) + kCtlCount, 0u);
    CHECK_HIP(hipGetLastError());
    int rc = read_ctl(ctx, kCtlCount, 1);
    if (rc) return rc;
    *S = ctx->h_ctl[kCtlCount];
    return MSCEER_OK;
}

CellGeom cell_geom(const Dims& d) {
    return CellGeom{(int64_t)d.Mx, (int64_t)d.My, (int64_t)d.Mz, (int64_t)d.Mx * (int64_t)d.My};
}

// Scratch of a family with S saddles: byte offsets of one buffer.
struct LineScratch {
    uint32_t W, chunks;  // lines of a window, chunks of the tape pool
    size_t keys, sorted, slots, pool, wmask, active, head, ended, lctl, tmp, tmp_bytes, bytes;
};

int line_scratch(uint32_t S, hipStream_t s, LineScratch* l) {
    const uint64_t nslots = 7ull * S;
    l->W = (uint32_t)std::min<uint64_t>(nslots, line_window());
    // tape pool: 128 slots per line of a window (volumes of noise and mixtures
    // record 20 to 40), at least 2^15 chunks
    l->chunks = env_size("MSCEER_LINE_CHUNKS", 1, kMaxChunks,
                         (uint32_t)std::min<uint64_t>(std::max<uint64_t>(2ull * l->W, 1u << 15), kMaxChunks));
    l->tmp_bytes = 0;
    CHECK_HIP(hipcub::DeviceRadixSort::SortKeysDescending(nullptr, l->tmp_bytes, (const uint64_t*)nullptr,
                                                          (uint64_t*)nullptr, (int)S, 0, 64, s));
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~(size_t)255;
        return at;
    };
    l->keys = take(8 * (size_t)S);
    l->sorted = take(8 * (size_t)S);
    l->slots = take(4 * nslots);
    l->pool = take(8 * (size_t)kTapeChunk * l->chunks);
    l->wmask = take(8 * (size_t)l->chunks);
    l->active = take((size_t)l->W * 4);
    l->head = take((size_t)l->W * 4);
    l->ended = take((size_t)l->W * 4);
    l->lctl = take(4 * kLcWords);
    l->tmp = take(l->tmp_bytes);
    l->bytes = off;
    return MSCEER_OK;
}

// The context's first set of tapes; where there is no memory for it, a second
// set kept by an earlier call makes room (nothing runs on it between calls).
int ensure_lines(msceer_ctx* ctx, size_t bytes) {
    if (ctx->lines.ensure(bytes) == hipSuccess) return MSCEER_OK;
    (void)hipGetLastError();
    ctx->lines2.release();
    CHECK_HIP(ctx->lines.ensure(bytes));
    return MSCEER_OK;
}

// Seeds and the first window's tapes of a family with S saddles, in buf (of
// the scratch's bytes), on stream s (the seeds by a scan, where the saddles are
// not listed, use the context's counter: then s is its stream).  The tapes of
// the first window read no label.
int begin_lines(msceer_ctx* ctx, const LineFamily& f, uint32_t S, const LineScratch& l, const DevBuf& buf, hipStream_t s,
                LineJob* job) {
    const VGrid g = make_vgrid(f.d.X, f.d.Y, f.d.Z);
    const CellGeom m = cell_geom(f.d);
    uint32_t* count = ctl_dev(ctx) + kCtlCount;
    const uint64_t nslots = 7ull * S;
    char* base = buf.as<char>();
    uint64_t* keys = (uint64_t*)(base + l.keys);
    uint64_t* sorted = (uint64_t*)(base + l.sorted);
    uint32_t* slots = (uint32_t*)(base + l.slots);
    uint32_t* lctl = (uint32_t*)(base + l.lctl);

    if (f.saddles) {
        hipLaunchKernelGGL(line_saddle_list_kernel, dim3(std::min<uint32_t>(blocks_for(S), 1024)), dim3(kThreads), 0, s,
                           *f.saddles, m, f.d.X, f.d.Y, f.values, f.asc ? 1 : 0, keys, S);
    } else {
        CHECK_HIP(launch_zero(count, 1, s));
        hipLaunchKernelGGL(line_saddles_kernel, dim3(2048), dim3(kThreads), 0, s, f.grad, m, f.d.X, f.d.Y, f.values,
                           f.asc ? 2 : 1, f.asc ? 1 : 0, keys, count, S);
    }
    CHECK_HIP(hipGetLastError());
    size_t tmp_bytes = l.tmp_bytes;
    CHECK_HIP(hipcub::DeviceRadixSort::SortKeysDescending(base + l.tmp, tmp_bytes, keys, sorted, (int)S, 0, 64, s));
    hipLaunchKernelGGL(line_seeds_kernel, dim3(blocks_for(S)), dim3(kThreads), 0, s, f.grad, m, sorted, S,
                       f.asc ? 1 : 0, slots);
    CHECK_HIP(hipGetLastError());

    LineArgs& a = job->a;
    a.src = GradSrc<double>{f.gradd};
    a.g = g;
    a.m = m;
    a.slots = slots;
    a.restr = f.restr;
    a.target = f.asc ? 4 : 5;
    a.asc = f.asc;
    a.gthr = (double)f.gthr;
    a.ethr = (double)f.ethr;
    a.max_iters = f.max_iters;
    a.pool = TapePool{(uint64_t*)(base + l.pool), l.chunks, lctl + kLcTop};
    a.wmask = (uint64_t*)(base + l.wmask);
    a.active = (uint32_t*)(base + l.active);
    a.head = (uint32_t*)(base + l.head);
    a.ended = (uint32_t*)(base + l.ended);
    a.stamp[0] = ctx->line_stamps.as<uint32_t>();
    a.stamp[1] = a.stamp[0] + f.d.cells;
    a.ctl = lctl;
    hipLaunchKernelGGL(line_ctl_init_kernel, dim3(1), dim3(64), 0, s, lctl, true);
    CHECK_HIP(hipGetLastError());

    job->nslots = nslots;
    job->W = l.W;
    return enqueue_tapes(a, 0, (uint32_t)std::min<uint64_t>(nslots, l.W), s);
}

// The rest of a family's lines, on the context's stream.
int finish_lines(msceer_ctx* ctx, const LineJob& job, LineStats* out) {
    hipStream_t s = ctx->stream;
    const LineArgs& a = job.a;
    const uint64_t nslots = job.nslots;
    const uint32_t W = job.W;
    uint32_t h[kLcWords];
    auto read_back = [&]() -> int {
        CHECK_HIP(hipMemcpyAsync(h, a.ctl, sizeof(h), hipMemcpyDeviceToHost, s));
        CHECK_HIP(hipStreamSynchronize(s));
        return MSCEER_OK;
    };
    const uint32_t max_rounds = env_size("MSCEER_LINE_ROUNDS", 2, kMaxRounds, kMaxRounds);
    const uint32_t group = std::min(8u, max_rounds);  // rounds between two read-backs
    uint32_t span = W;  // lines of the next window
    uint64_t w0 = 0;
    while (w0 < nslots) {
        const uint32_t a0 = (uint32_t)w0;
        const uint32_t w1 = (uint32_t)std::min<uint64_t>(nslots, w0 + span);
        const uint32_t n = w1 - a0;
        if (ctx->line_tag <= kMaxRounds) {
            hipLaunchKernelGGL(line_fill_kernel, dim3(2048), dim3(kThreads), 0, s, a.stamp[0],
                               (uint64_t)(ctx->line_stamps.bytes / 4), kNoLine);
            CHECK_HIP(hipGetLastError());
            ctx->line_tag = kTopTag;
        }
        const uint32_t wave_blocks = std::min<uint32_t>(blocks_for((uint64_t)n * 64), 2048);
        if (w0 > 0) {
            int rc = enqueue_tapes(a, a0, w1, s);
            if (rc) return rc;
        }
        out->windows++;
        // rounds in groups; the host reads back only whether the last one
        // still changed a line (then the commit behind it did nothing)
        uint32_t round = 0;
        uint32_t cut = 0;
        while (true) {
            for (uint32_t j = 0; j < group; j++, round++)
                hipLaunchKernelGGL(line_round_kernel, dim3(wave_blocks), dim3(kThreads), 0, s, a, a0, w1, round,
                                   ctx->line_tag--);
            hipLaunchKernelGGL(line_commit_kernel, dim3(wave_blocks), dim3(kThreads), 0, s, a, a0, w1, round - 1, true);
            CHECK_HIP(hipGetLastError());
            int rc = read_back();
            if (rc) return rc;
            const uint32_t wc = std::min(h[kLcOverflow], w1);  // lines of this window
            if (h[kLcChanged + (round - 1) % 3] == 0) {
                cut = wc;
                if (wc < w1) out->overflows++;
                break;
            }
            if (round + group > max_rounds) {
                // the lines before the lowest one still changing are exact
                cut = h[kLcLowest + (round - 1) % 3];
                hipLaunchKernelGGL(line_commit_kernel, dim3(wave_blocks), dim3(kThreads), 0, s, a, a0, cut, 0u, false);
                CHECK_HIP(hipGetLastError());
                out->cuts++;
                break;
            }
        }
        out->rounds += round;
        // The lines from the cut on were traced for nothing: the next window
        // takes no more than this one could resolve, or half of it (the pool
        // is shared out as the lanes come, so an early line can be the one
        // without room).  It doubles again where its tapes filled at most two
        // fifths of the pool and its rounds ended early.  (28x30x260 ridges, a
        // pool of 1500 chunks where 26000 are wanted: 44591 streamlines traced
        // for 15912; with windows as long as before, 25.4 million.)
        if (cut < w1) span = std::max(cut - a0, std::max(n / 2, 1u));
        else if (5ull * h[kLcTop] <= 2ull * a.pool.chunks && round <= max_rounds / 4)
            span = (uint32_t)std::min<uint64_t>(W, 2ull * span);
        if (cut == a0) {
            // the first line's tape did not fit the pool: it alone, in order
            hipLaunchKernelGGL(line_direct_kernel, dim3(1), dim3(64), 0, s, a, a0);
            CHECK_HIP(hipGetLastError());
            out->direct++;
            w0 = a0 + 1;
            continue;
        }
        w0 = cut;
    }
    int rc = read_back();
    if (rc) return rc;
    out->traced = h[kLcTraced];
    out->replayed = h[kLcCut];
    out->voxels = h[kLcVoxels];
    return MSCEER_OK;
}


}  // namespace

// A second family's tapes are traced on another stream beside the first's: the
// tape kernels last as long as their longest streamlines and leave most of the
// chip idle (256^3 mixture: 2.4 and 3.0 ms one after the other).  The labels
// are still resolved one family after the other.  The first family's set of
// tapes is allocated first; without memory for a second one the families take
// turns with it.
int run_lines(msceer_ctx* ctx, const LineFamily* families, int n, LineStats* out) {
    hipStream_t s = ctx->stream;
    LineJob jobs[2];
    LineScratch scratch[2] = {};
    uint32_t S[2] = {0, 0};
    bool begun[2] = {false, false};
    for (int i = 0; i < n; i++) {
        const Dims& d = families[i].d;
        if (d.cells >= 0xFFFFFFFFull) return MSCEER_ETOOBIG;
        int rc = count_saddles(ctx, families[i], cell_geom(d), &S[i]);
        if (rc) return rc;
        out[i].saddles = S[i];
        if ((uint64_t)S[i] * 7 >= 0xFFFFFFFFull) return MSCEER_ETOOBIG;
        // two stamps per cell, refilled when they are new or the tags run out
        if (ctx->line_stamps.bytes < 8 * d.cells) ctx->line_tag = 0;
        if (S[i] == 0) continue;
        CHECK_HIP(ctx->line_stamps.ensure(8 * d.cells));
        rc = line_scratch(S[i], s, &scratch[i]);
        if (rc) return rc;
    }
    // whatever happens, nothing is left running on the second stream
    struct Join {
        msceer_ctx* ctx;
        bool on = false;
        ~Join() {
            if (on) (void)hipStreamSynchronize(ctx->side);
        }
    } join{ctx};
    if (n == 2 && S[0] && S[1] && families[1].saddles) {
        const int rc = ensure_lines(ctx, scratch[0].bytes);
        if (rc) return rc;
        if (!ctx->side) CHECK_HIP(hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking));
        if (!ctx->side_ev) CHECK_HIP(hipEventCreateWithFlags(&ctx->side_ev, hipEventDisableTiming));
        CHECK_HIP(hipEventRecord(ctx->side_ev, s));
        CHECK_HIP(hipStreamWaitEvent(ctx->side, ctx->side_ev, 0));
        join.on = true;
        begun[1] = ctx->lines2.ensure(scratch[1].bytes) == hipSuccess &&
                   begin_lines(ctx, families[1], S[1], scratch[1], ctx->lines2, ctx->side, &jobs[1]) == MSCEER_OK;
        if (!begun[1]) {
            (void)hipGetLastError();
            CHECK_HIP(hipStreamSynchronize(ctx->side));
            ctx->lines2.release();
            jobs[1] = LineJob{};
        }
    }
    for (int i = 0; i < n; i++) {
        if (S[i] == 0) continue;
        int rc;
        if (begun[i]) {
            CHECK_HIP(hipEventRecord(ctx->side_ev, ctx->side));
            CHECK_HIP(hipStreamWaitEvent(s, ctx->side_ev, 0));
        } else {
            rc = ensure_lines(ctx, scratch[i].bytes);
            if (rc) return rc;
            rc = begin_lines(ctx, families[i], S[i], scratch[i], ctx->lines, s, &jobs[i]);
            if (rc) return rc;
        }
        rc = finish_lines(ctx, jobs[i], &out[i]);
        if (rc) return rc;
    }
    join.on = false;  // (the context's stream has waited for it)
    return MSCEER_OK;
}

}  // namespace msceer
