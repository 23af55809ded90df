// The 1-manifolds' order realised a second way (test infrastructure):
// speculative traces over windows of streamlines with footprints, and replay,
// in order, of the components of those that interact, as label policies of the
// kernels' own trace (lines_core.hpp).
#pragma once

#include "lines_core.hpp"

namespace msceer {
namespace {

// Footprints: every cell a speculative trace tests or labels, appended (with
// repeats) to chunks of a shared pool, one chain per line (and a second chain
// of the cells it labelled): chunk = the index of the next chunk (or kNoLine)
// and kChunk - 1 cells, the last chunk of a footprint ended by kNoLine.
constexpr uint32_t kChunk = 32;

struct Pool {
    uint32_t* cells;     // capacity words
    uint32_t capacity;   // a multiple of kChunk
    uint32_t* top;       // next free word
};

// Speculation: committed labels plus the line's own labels, known exactly
// (own[c]: the last line of the window that labelled c; its second chain
// where another line overwrote that mark).  Labelled cells claim wstamp (the
// lowest line of the window labelling them); the first claim of a cell
// appends it to the window's list of labelled cells.
struct SpecLabels {
    const int8_t* restr;
    int8_t target;
    uint32_t* wstamp;
    uint32_t* pstamp;
    uint32_t* own;
    uint32_t line;
    Pool pool;
    uint32_t* touched;     // cells labelled (or possibly labelled) in the window
    uint32_t* ntouched;
    struct Chain {
        uint32_t head = kNoLine, chunk = kNoLine, fill = 0;
    } all, wrote, maybe;   // the footprint; the cells labelled; the cells a stop could label
    uint32_t last[6];      // the cells of the last stop_here, not recorded again
    int nlast = -1;
    bool over = false;
    __device__ void append(Chain& ch, uint32_t c) {
        if (over) return;
        if (ch.chunk == kNoLine || ch.fill == kChunk - 1) {
            const uint32_t at = atomicAdd(pool.top, kChunk);
            if (at + kChunk > pool.capacity) {
                over = true;
                return;
            }
            pool.cells[at] = kNoLine;
            if (ch.chunk == kNoLine) ch.head = at;
            else pool.cells[ch.chunk] = at;
            ch.chunk = at;
            ch.fill = 0;
        }
        pool.cells[ch.chunk + 1 + ch.fill] = c;
        ch.fill++;
    }
    __device__ void claim(uint32_t* stamp, uint32_t c) {
        if (atomicMin(&stamp[c], line) == kNoLine) {
            const uint32_t at = atomicAdd(ntouched, 1u);
            if (at < pool.capacity) touched[at] = c;  // (never more cells than pool words)
        }
    }
    // Did this line label c?  own[c] says yes unless another line of the
    // window labelled c since; wstamp[c] > line says no (a line's own claim
    // keeps wstamp at or below it); otherwise the line's labels are searched.
    __device__ bool mine(uint32_t c) const {
        if (own[c] == line) return true;
        if (wstamp[c] > line) return false;
        for (uint32_t ch = wrote.head; ch != kNoLine; ch = pool.cells[ch]) {
            const uint32_t n = ch == wrote.chunk ? wrote.fill : kChunk - 1;
            for (uint32_t j = 0; j < n; j++)
                if (pool.cells[ch + 1 + j] == c) return true;
        }
        return false;
    }
    __device__ bool test(uint32_t c) {
        append(all, c);
        return restr[c] == target || mine(c);
    }
    __device__ void write(uint32_t c) {
        append(all, c);
        append(wrote, c);
        if (over) return;  // the window ends before this line
        own[c] = line;
        claim(wstamp, c);
    }
    // Cells a stop at this point would label (its digitization start ->
    // here): footprint, and claimed in pstamp, so that a replay stopping here
    // stays within what the speculation saw.
    __device__ void stop_here(const CellGeom& m, const V3<double>& a, const V3<double>& b, bool asc) {
        uint32_t cells[6];
        const int n = digitize_cells(m, a, b, asc, cells);
        bool same = n == nlast;
        for (int k = 0; same && k < n; k++) same = cells[k] == last[k];
        if (same) return;
        nlast = n;
        for (int k = 0; k < n; k++) {
            last[k] = cells[k];
            append(all, cells[k]);
            append(maybe, cells[k]);
            if (over) return;
            claim(pstamp, cells[k]);
        }
    }
    __device__ void leave() {}
    // End marks of the last chunks.
    __device__ void finish() {
        if (over) return;
        if (all.chunk != kNoLine && all.fill < kChunk - 1) pool.cells[all.chunk + 1 + all.fill] = kNoLine;
        if (wrote.chunk != kNoLine && wrote.fill < kChunk - 1) pool.cells[wrote.chunk + 1 + wrote.fill] = kNoLine;
        if (maybe.chunk != kNoLine && maybe.fill < kChunk - 1) pool.cells[maybe.chunk + 1 + maybe.fill] = kNoLine;
    }
    __device__ bool ok() const { return !over; }
};

// Union-find over the lines of a window (relative indices).
__device__ __forceinline__ uint32_t lf_parent(uint32_t* p, uint32_t x) {
    return __hip_atomic_load(&p[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t lf_find(uint32_t* p, uint32_t x) {
    uint32_t q = lf_parent(p, x);
    while (q != x) {
        const uint32_t gq = lf_parent(p, q);
        if (gq != q) __hip_atomic_store(&p[x], gq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = q;
        q = gq;
    }
    return x;
}
// Hook the later root under the earlier one, so a component's root is its
// first line.
__device__ void lf_union(uint32_t* p, uint32_t a, uint32_t b) {
    while (true) {
        a = lf_find(p, a);
        b = lf_find(p, b);
        if (a == b) return;
        if (a > b) { const uint32_t t = a; a = b; b = t; }
        uint32_t expected = b;
        if (__hip_atomic_compare_exchange_strong(&p[b], &expected, a, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
    }
}

// Replay of one component, its lines in order: committed labels plus those
// its earlier lines gave (lstamp).  A cell that lines of the window labelled,
// or could label by stopping, in speculation belongs to their component; a
// replayed line may test it only in its own component, and may label only
// cells it labelled, or could label, itself in speculation.  Anything else
// means the line went beyond what the speculation saw, and the window is cut
// before it.
struct ReplayLabels {
    const int8_t* restr;
    int8_t target;
    const uint32_t* wstamp;
    const uint32_t* pstamp;
    uint32_t* lstamp;
    const uint32_t* own;
    const uint32_t* pool;
    uint32_t whead, mhead;  // chains of the cells this line labelled / a stop could label, in speculation
    uint32_t* parent;
    uint32_t w0, wc, root, line;
    uint32_t* why;          // failure counters: [0] tests, [1] labels
    bool bad;
    __device__ static bool in_chain(const uint32_t* pool, uint32_t head, uint32_t c) {
        for (uint32_t ch = head; ch != kNoLine; ch = pool[ch])
            for (uint32_t j = 1; j < kChunk; j++) {
                const uint32_t x = pool[ch + j];
                if (x == kNoLine) break;
                if (x == c) return true;
            }
        return false;
    }
    __device__ bool foreign(uint32_t w) const { return w >= w0 && w < wc && lf_find(parent, w - w0) != root; }
    __device__ bool test(uint32_t c) {
        if (foreign(wstamp[c]) || foreign(pstamp[c])) {
            if (!bad) atomicAdd(&why[0], 1u);
            bad = true;
            return false;
        }
        return restr[c] == target || lstamp[c] != kNoLine;
    }
    __device__ void write(uint32_t c) {
        const bool seen = own[c] == line || (wstamp[c] <= line && in_chain(pool, whead, c)) ||
                          (pstamp[c] <= line && in_chain(pool, mhead, c));
        if (!seen) {
            if (!bad) atomicAdd(&why[1], 1u);
            bad = true;
            return;
        }
        lstamp[c] = line;
    }
    __device__ bool ok() const { return !bad; }
    __device__ void stop_here(const CellGeom&, const V3<double>&, const V3<double>&, bool) {}
    __device__ void leave() {}
};

}  // namespace
}  // namespace msceer
