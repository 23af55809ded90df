// Device code of the accurate 1-manifolds (lines.hip): cell geometry, the
// saddles' seed search, one digitizing streamline, its trace in order against
// the labels and its tape, and a tape's evaluation.  Kept in a header so that a
// host build of the same source can be checked against the CPU oracle; the
// includer provides what tracer.hpp needs plus atomicAdd.
#pragma once

#include "tracer.hpp"

#pragma clang fp contract(off)

namespace msceer {
namespace {

constexpr uint32_t kNoLine = 0xFFFFFFFFu;
constexpr int kAbort = 100;  // trace event: the label policy stopped it (a tape beyond the pool)

struct CellGeom {
    int64_t Mx, My, Mz, sxy;
    __device__ uint32_t id(int64_t x, int64_t y, int64_t z) const { return (uint32_t)(x + Mx * (y + My * z)); }
    __device__ void xyz(uint32_t c, int64_t& x, int64_t& y, int64_t& z) const {
        x = (int64_t)c % Mx;
        y = ((int64_t)c / Mx) % My;
        z = (int64_t)c / sxy;
    }
    __device__ int64_t off(int a) const { return a == 0 ? 1 : (a == 1 ? Mx : sxy); }
    __device__ int64_t ext(int a) const { return a == 0 ? Mx : (a == 1 ? My : Mz); }
    // Cell coordinates inside the complex.  A streamline away from the
    // boundary stays inside; this only keeps a step that a huge error
    // threshold let run far from addressing outside the arrays.
    __device__ bool inside(int64_t x, int64_t y, int64_t z) const {
        return x >= 0 && y >= 0 && z >= 0 && x < Mx && y < My && z < Mz;
    }
    // the same for coordinates from cell_floor (an id has 32 bits, an extent 17)
    __device__ __forceinline__ uint32_t id32(int x, int y, int z) const {
        return (uint32_t)x + (uint32_t)Mx * ((uint32_t)y + (uint32_t)My * (uint32_t)z);
    }
    __device__ __forceinline__ bool inside32(int x, int y, int z) const {
        return (uint32_t)x < (uint32_t)Mx && (uint32_t)y < (uint32_t)My && (uint32_t)z < (uint32_t)Mz;
    }
};

// floor(v), cut off far outside any volume so that twice it fits an int.
__device__ __forceinline__ int cell_floor(double v) {
    const int f = (int)floor(v);
    return f < -(1 << 29) ? -(1 << 29) : (f > (1 << 29) ? 1 << 29 : f);
}

// Order key of a float: monotone, -0 and +0 equal (as float comparison has them).
__device__ __forceinline__ uint32_t value_key(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) == 0u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ bool critical(const uint8_t* grad, uint32_t c) { return ((grad[c] >> 2) & 7u) == 7u; }

__device__ __forceinline__ uint32_t pair_of(const CellGeom& m, const uint8_t* grad, uint32_t c) {
    const uint32_t code = (grad[c] >> 2) & 7u;
    const int64_t o = m.off((int)(code >> 1));
    return (uint32_t)((int64_t)c + ((code & 1u) ? -o : o));
}

__device__ __forceinline__ double comp(const V3<double>& v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }

// DigitizeSegmentInternal: the faces the segment a -> b crosses, by their
// crossing parameter; for each face that bounds the current cell, the
// current cell and the face, then the cell beyond becomes current.  ASC:
// voxel faces, cells = hexes; DSC: the dual grid (positions shifted by half a
// voxel), faces = edges, cells = vertices.  digitize_cells lists those cells
// in order (cell, face, cell, face, ...: at most six) without looking at any
// label; digitize labels them in that order and stops at the first one that
// already carries the target.
__device__ __forceinline__ int digitize_cells(const CellGeom& m, V3<double> a, V3<double> b, bool asc, uint32_t* out) {
    if (!asc) {
        a = {a.x + 0.5, a.y + 0.5, a.z + 0.5};
        b = {b.x + 0.5, b.y + 0.5, b.z + 0.5};
    }
    const V3<double> ab{b.x - a.x, b.y - a.y, b.z - a.z};
    // the faces crossed, at most one per axis; every index below is known when
    // compiled, so they stay in registers, and the faces' coordinates are kept
    // (from the id they cost two divisions each)
    uint32_t face[3] = {};
    double tc[3] = {};
    int p[3][3] = {};
    int n = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double av = comp(a, d), bv = comp(b, d);
        const int va = (int)floor(av), vb = (int)floor(bv);
        if (va == vb) continue;
        const int plane = va > vb ? va : vb;
        const double t = ((double)plane - av) / (bv - av);
        if (t < 0 || t > 1) return 0;
        int fc[3];
#pragma unroll
        for (int k = 0; k < 3; k++)
            fc[k] = 2 * cell_floor(comp(ab, k) * t + comp(a, k)) + (k == d ? 0 : 1) - (asc ? 0 : 1);
        if (!m.inside32(fc[0], fc[1], fc[2])) return 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i == n) {
                tc[i] = t;
                face[i] = m.id32(fc[0], fc[1], fc[2]);
                for (int k = 0; k < 3; k++) p[i][k] = fc[k];
            }
        n++;
    }
    if (n == 0) return 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = i + 1; j < 3; j++)
            if (j < n && tc[i] > tc[j]) {
                const uint32_t tf = face[i]; face[i] = face[j]; face[j] = tf;
                const double tt = tc[i]; tc[i] = tc[j]; tc[j] = tt;
                for (int k = 0; k < 3; k++) { const int tp = p[i][k]; p[i][k] = p[j][k]; p[j][k] = tp; }
            }
    const int s0 = 2 * cell_floor(a.x) + (asc ? 1 : 0), s1 = 2 * cell_floor(a.y) + (asc ? 1 : 0),
              s2 = 2 * cell_floor(a.z) + (asc ? 1 : 0);
    if (!m.inside32(s0, s1, s2)) return 0;
    uint32_t cur = m.id32(s0, s1, s2);
    int k = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (i >= n) continue;
        bool has = false;
        uint32_t next = cur;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (asc ? (p[i][d] & 1) != 0 : (p[i][d] & 1) == 0) continue;
            if (p[i][d] < (int)m.ext(d) - 1) {
                const uint32_t c = face[i] + (uint32_t)m.off(d);
                if (c == cur) has = true; else next = c;
            }
            if (p[i][d] > 0) {
                const uint32_t c = face[i] - (uint32_t)m.off(d);
                if (c == cur) has = true; else next = c;
            }
        }
        if (!has) continue;
#pragma unroll
        for (int q = 0; q < 3; q++)
            if (k == 2 * q) {
                out[2 * q] = cur;
                out[2 * q + 1] = face[i];
            }
        k += 2;
        cur = next;
    }
    return k;
}

// cells[k] of digitize_cells, by selects.
__device__ __forceinline__ uint32_t pick6(const uint32_t* cells, int k) {
    const uint32_t c0 = cells[0], c1 = cells[1], c2 = cells[2], c3 = cells[3], c4 = cells[4], c5 = cells[5];
    const uint32_t lo = k == 0 ? c0 : (k == 1 ? c1 : c2), hi = k == 3 ? c3 : (k == 4 ? c4 : c5);
    return k < 3 ? lo : hi;
}

// The seed cells of saddle s from the short V-path search
// (ondemandaccurate.cxx:319-351 ASC, 448-480 DSC), at most six, in out[0..5]
// (kNoLine where absent), and the saddle in out[6].  The search pops at most
// five cells: the saddle, whose two cofacets (ASC) / facets (DSC) are new,
// then cells that each add one new neighbour.
__device__ inline void saddle_seeds(const uint8_t* grad, const CellGeom& m, uint32_t s, bool asc, uint32_t* out) {
    uint32_t result[6], queue[6], seen[16];
    int nres = 0, qh = 0, qt = 0, ns = 0;
    auto is_seen = [&](uint32_t c) {
        for (int i = 0; i < ns; i++)
            if (seen[i] == c) return true;
        return false;
    };
    queue[qt++] = s;
    for (int counter = 4; qh < qt && counter >= 0; counter--) {
        const uint32_t cur = queue[qh++];
        if (!is_seen(cur) && ns < 16) seen[ns++] = cur;
        int64_t p[3];
        m.xyz(cur, p[0], p[1], p[2]);
        for (int a = 0; a < 3; a++) {
            if (asc ? (p[a] & 1) != 0 : (p[a] & 1) == 0) continue;
            for (int sg = 0; sg < 2; sg++) {
                if (sg == 0 ? p[a] >= m.ext(a) - 1 : p[a] <= 0) continue;
                const uint32_t t = (uint32_t)((int64_t)cur + (sg == 0 ? m.off(a) : -m.off(a)));
                if (is_seen(t)) continue;
                if (nres < 6) result[nres++] = t;
                if (ns < 16) seen[ns++] = t;
                if (!critical(grad, t)) {
                    const uint32_t pr = pair_of(m, grad, t);
                    if (ns < 16) seen[ns++] = pr;
                    if (qt < 6) queue[qt++] = pr;
                }
            }
        }
    }
    for (int j = 0; j < 6; j++) out[j] = j < nres ? result[j] : kNoLine;
    out[6] = s;
}

// ---- one streamline ----------------------------------------------------------

// Label policies of a trace: test(c) -- does cell c carry the target (a
// checker or digitizing test); write(c) -- give it the target; stop_here() --
// a test at a step inside a voxel follows, where a stop digitizes no further
// than that step; leave() -- one at the step out of it; ok() -- false once the
// trace must stop for the policy's own reasons.

// Alone and in order: the restriction labels themselves.
struct DirectLabels {
    int8_t* restr;
    int8_t target;
    __device__ bool test(uint32_t c) { return restr[c] == target; }
    __device__ void write(uint32_t c) { restr[c] = target; }
    __device__ bool ok() const { return true; }
    __device__ void stop_here(const CellGeom&, const V3<double>&, const V3<double>&, bool) {}
    __device__ void leave() {}
};

// ---- tapes -------------------------------------------------------------------
//
// The path of a streamline depends on no label: labels only decide where it
// stops and which of the cells it digitizes it reaches.  A tape is the
// sequence of what a streamline would ask of the labels if nothing but its own
// labels stopped it, and what the line does in the reference's order follows
// from the tape and the labels other lines give alone (tape_chunk), without
// tracing again.  Entries, 64 bits each: the cell (low word), and in the high
// word the kind, the first-of-a-list flag and the slot of the line's previous
// list entry of the same cell.
//   kStay   a stop test at a step that stays in its voxel; the list of kStop
//           entries behind it is what a stop there digitizes
//   kExit   a stop test at the step that leaves a voxel; the kList entries
//           behind it are digitized whether it stops or not
//   kList   a digitized cell (in lists: the first labelled cell ends a list)
//   kStop   as kList, applied only if the kStay test before them stops
// A test repeated with no list entry of its cell in between asks the same
// question again and is not recorded.  The first cell of a list carries the
// target once the list is done (it had it, or takes it), so a test of a cell
// that was first in an earlier list stops the line whatever other lines do:
// the tape ends there (history: the last kHistory such cells; an older one
// only makes the tape longer than it need be).
// Tapes are chains of chunks of 64 slots: slot 0 holds the next chunk (low
// word) and the number of entries (high word), slots 1.. the entries.
constexpr uint32_t kStay = 0, kExit = 1, kList = 2, kStop = 3;
constexpr int kKindShift = 29;
constexpr uint32_t kFirst = 0x80000000u;     // first entry of a list
constexpr uint32_t kNoPrev = 0x1FFFFFFFu;    // no earlier kList entry of the cell
constexpr uint32_t kTapeChunk = 64;          // slots of a chunk
constexpr uint32_t kMaxTapeChunks = 1024;    // chunks of one tape (longer lines are traced alone, in order)
constexpr uint32_t kHistory = 32;

struct TapePool {
    uint64_t* slots;    // chunks * kTapeChunk
    uint32_t chunks;
    uint32_t* top;      // next free chunk
};

// Recording policy of a trace.  hist: kHistory words, hstride apart.
struct TapeLabels {
    const int8_t* restr;
    int8_t target;
    bool committed;      // earlier windows have labelled cells: a test of one ends the tape
    TapePool pool;
    uint32_t* hist;
    uint32_t hstride;
    uint32_t nhist = 0, last = kNoLine;
    uint32_t head = kNoLine, chunk = kNoLine, fill = 0, nchunks = 0;
    bool over = false, staying = false, asc = false;
    CellGeom geom{};
    V3<double> from{}, to{};
    // first: the first entry of a list
    __device__ __forceinline__ void append(uint32_t kind, uint32_t c, bool first = false) {
        if (over) return;
        if (chunk == kNoLine || fill == kTapeChunk - 1) {
            const uint32_t at = nchunks < kMaxTapeChunks ? atomicAdd(pool.top, 1u) : kNoLine;
            if (at >= pool.chunks) {
                over = true;
                return;
            }
            if (chunk == kNoLine) head = at;
            else pool.slots[(uint64_t)chunk * kTapeChunk] = (uint64_t)fill << 32 | at;
            chunk = at;
            fill = 0;
            nchunks++;
        }
        fill++;
        pool.slots[(uint64_t)chunk * kTapeChunk + fill] =
            (uint64_t)(kind << kKindShift | kNoPrev | (first ? kFirst : 0u)) << 32 | c;
    }
    __device__ __forceinline__ void finish() {
        if (!over && chunk != kNoLine) pool.slots[(uint64_t)chunk * kTapeChunk] = (uint64_t)fill << 32 | kNoLine;
    }
    __device__ __forceinline__ void stop_here(const CellGeom& m, const V3<double>& a, const V3<double>& b, bool up) {
        staying = true;
        geom = m;
        from = a;
        to = b;
        asc = up;
    }
    __device__ __forceinline__ void leave() { staying = false; }
    __device__ __forceinline__ bool test(uint32_t c) {
        if (c == last) return false;
        last = c;
        append(staying ? kStay : kExit, c);
        if (staying) {
            uint32_t cells[6] = {};
            const int n = digitize_cells(geom, from, to, asc, cells);
#pragma unroll 1
            for (int k = 0; k < n; k++) append(kStop, pick6(cells, k), k == 0);
        }
        bool hit = committed && restr[c] == target;
        const uint32_t n = nhist < kHistory ? nhist : kHistory;
        // (reads of eight words in flight at a time; those beyond n count for nothing)
        for (uint32_t k = 0; k < n; k += 8) {
            uint32_t h[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; j++) h[j] = hist[(k + j) * hstride];
#pragma unroll
            for (uint32_t j = 0; j < 8; j++) hit |= (h[j] == c) & (k + j < n);
        }
        return hit;
    }
    __device__ __forceinline__ void list(const uint32_t* cells, int n) {
#pragma unroll 1
        for (int k = 0; k < n; k++) {
            const uint32_t c = pick6(cells, k);
            append(kList, c, k == 0);
            if (c == last) last = kNoLine;
        }
        // an exit without a list: the next test is recorded again, so that no
        // later list is taken for this exit's
        if (n > 0) hist[(nhist++ % kHistory) * hstride] = cells[0];
        else last = kNoLine;
    }
    __device__ __forceinline__ bool ok() const { return !over; }
};

__device__ __forceinline__ void digitize(const CellGeom& m, const V3<double>& a, const V3<double>& b, bool asc, TapeLabels& lab) {
    uint32_t cells[6] = {};
    const int n = digitize_cells(m, a, b, asc, cells);
    lab.list(cells, n);
}

// What a line does along its tape, chunk by chunk.
struct TapeState {
    bool broken = false;   // the list at hand met a labelled cell
    uint32_t ending = 0;   // a test stopped the line: 1 its kStop list, 2 its kList list remains
    bool begun = false;    // that list has begun
};

// Evaluates the entries of one chunk (bit k of a mask: slot k).  test /
// exitm / stopm / first: kinds (neither test nor stopm: kList); lab: cells
// that carry the target for this line (committed, or given by an earlier
// line); prevm: entries with an earlier list entry of the same cell, whose
// bit own(k, w) returns.  Returns the list entries whose cell carries the
// target after them -- reached (labelled already, or labelled now) or
// labelled by the line before; *stop: the slot at which the line ended, 0 if
// it goes on.
template <class Own>
__device__ inline uint64_t tape_chunk(TapeState& s, uint32_t n, uint64_t test, uint64_t exitm, uint64_t stopm,
                                      uint64_t first, uint64_t lab, uint64_t prevm, Own own, uint32_t* stop) {
    const uint64_t all = n >= 63 ? ~1ull : ((1ull << (n + 1)) - 2ull);
    *stop = 0;
    if (!((lab | prevm) & all) && s.ending == 0 && !s.broken) return all & ~test & ~stopm;
    uint64_t w = 0;
    for (uint32_t k = 1; k <= n; k++) {
        const uint64_t bit = 1ull << k;
        const bool is_test = (test & bit) != 0, is_stop = (stopm & bit) != 0, is_first = (first & bit) != 0;
        if (s.ending) {
            const bool belongs = !is_test && (s.begun ? !is_first : (is_first && is_stop == (s.ending == 1)));
            if (!belongs) {
                *stop = k;
                return w;
            }
            s.begun = true;
        }
        const bool mine = (prevm & bit) && own(k, w);
        const bool labelled = (lab & bit) || mine;
        if (is_test) {
            if (labelled) {
                s.ending = (exitm & bit) ? 2u : 1u;
                s.begun = false;
            }
            continue;
        }
        if (is_first) s.broken = false;
        if (is_stop && s.ending != 1) {
            if (mine) w |= bit;
            continue;
        }
        if (!s.broken || mine) w |= bit;
        if (labelled) s.broken = true;
    }
    return w;
}

// Label the cells of digitize_cells in order; stop at the first one that
// already carries the target.
template <class L>
__device__ __forceinline__ void digitize(const CellGeom& m, const V3<double>& a, const V3<double>& b, bool asc, L& lab) {
    uint32_t cells[6] = {};
    const int n = digitize_cells(m, a, b, asc, cells);
    for (int k = 0; k < n; k++) {
        const uint32_t c = pick6(cells, k);
        if (lab.test(c)) return;
        lab.write(c);
        if (!lab.ok()) return;
    }
}

template <class L>
__device__ __forceinline__ int advect_voxel(const VGrid& g, const CellGeom& m, Tracer<double>& t, const V3<double>& start, double dir,
                            double gthr, double ethr, bool asc, L& lab) {
    while (true) {
        if (!(t.iters-- > 0)) return kOverMax;
        if (!(t.old.x == t.cur.x && t.old.y == t.cur.y && t.old.z == t.cur.z)) {
            if ((int)t.cur.x != (int)t.old.x || (int)t.cur.y != (int)t.old.y || (int)t.cur.z != (int)t.old.z)
                return kOutOfVoxel;
            t.gr = trilin(t.c, t.cur.x - (double)t.bx, t.cur.y - (double)t.by, t.cur.z - (double)t.bz);
            t.gm = sqrt(t.gr.x * t.gr.x + t.gr.y * t.gr.y + t.gr.z * t.gr.z);
            if (t.gm * t.step > kMaxStep) t.step = kMaxStep / t.gm;
            t.old = t.cur;
        }
        if (t.gm < gthr) return kLowGradient;
        const double s = dir * t.step, hs = (dir * 0.5) * t.step;
        const V3<double> full{t.gr.x * s, t.gr.y * s, t.gr.z * s};
        const V3<double> half{t.gr.x * hs, t.gr.y * hs, t.gr.z * hs};
        const V3<double> hg = trilin(t.c, t.cur.x + half.x - (double)t.bx, t.cur.y + half.y - (double)t.by,
                                     t.cur.z + half.z - (double)t.bz);
        const V3<double> two{hg.x * hs + half.x, hg.y * hs + half.y, hg.z * hs + half.z};
        const double dx = two.x - full.x, dy = two.y - full.y, dz = two.z - full.z;
        const double err = dx * dx + dy * dy + dz * dz;
        if (!(err < ethr)) {
            t.step = t.step * 0.5;
            continue;
        }
        t.cur = {t.cur.x + two.x, t.cur.y + two.y, t.cur.z + two.z};
        if (t.near) { t.cur.x = clampc(t.cur.x, g.X); t.cur.y = clampc(t.cur.y, g.Y); t.cur.z = clampc(t.cur.z, g.Z); }
        const double grow = t.step * 1.8, cap = kMaxStep / t.gm;
        t.step = grow < cap ? grow : cap;
        if (t.near) return kHitPreassigned;
        // a stop at a step that stays in the voxel digitizes start -> here
        // instead of the whole voxel segment
        if ((int)t.cur.x == (int)t.old.x && (int)t.cur.y == (int)t.old.y && (int)t.cur.z == (int)t.old.z)
            lab.stop_here(m, start, t.cur, asc);
        else
            lab.leave();
        const int cx = asc ? 2 * cell_floor(t.cur.x) + 1 : 2 * cell_floor(t.cur.x + 0.5);
        const int cy = asc ? 2 * cell_floor(t.cur.y) + 1 : 2 * cell_floor(t.cur.y + 0.5);
        const int cz = asc ? 2 * cell_floor(t.cur.z) + 1 : 2 * cell_floor(t.cur.z + 0.5);
        if (!m.inside32(cx, cy, cz)) continue;
        const bool hit = lab.test(m.id32(cx, cy, cz));
        if (!lab.ok()) return kAbort;
        if (hit) return kHitPreassigned;
    }
}

// IntegrateStreamline from the centre of seed cell `seed` (cell coordinates / 2).
template <class L>
__device__ __forceinline__ int trace_line(const GradSrc<double>& src, const VGrid& g, const CellGeom& m, uint32_t seed, bool asc,
                          double gthr, double ethr, int max_iters, L& lab, uint32_t* voxels) {
    int64_t sx, sy, sz;
    m.xyz(seed, sx, sy, sz);
    Tracer<double> t;
    t.cur = {(double)sx * 0.5, (double)sy * 0.5, (double)sz * 0.5};
    t.iters = max_iters;
    tracer_load(src, g, t, (int)(t.cur.x + 0.5), (int)(t.cur.y + 0.5), (int)(t.cur.z + 0.5));
    tracer_begin(t);
    const double dir = asc ? 1.0 : -1.0;
    while (true) {
        const V3<double> start = t.cur;
        const int ev = advect_voxel(g, m, t, start, dir, gthr, ethr, asc, lab);
        (*voxels)++;
        if (ev == kAbort) return kAbort;
        if (!t.near) {
            digitize(m, start, t.cur, asc, lab);
            if (!lab.ok()) return kAbort;
        }
        if (ev != kOutOfVoxel) return ev;
        int x, y, z;
        nearest_xyz(g, t.cur, t.near, x, y, z);
        tracer_load(src, g, t, x, y, z);
        tracer_begin(t);
    }
}

}  // namespace
}  // namespace msceer
