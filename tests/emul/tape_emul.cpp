// Host emulation of the 1-manifold tapes (test infrastructure): the tape
// recording and the chunk evaluation of lines_core.hpp, the code the gfx950
// kernels run, driven on the CPU -- a tape per line of a window, links to the
// earlier list entries of a cell, rounds in which every line is evaluated
// against the labels the lines gave in the round before until none changes,
// commit -- and compared with the oracle's one-thread saddle loops.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <unordered_map>
#include <vector>

// what the HIP build provides to the device headers
#define __host__
#define __device__
#define __forceinline__ inline
#define __restrict__
#define __HIP_MEMORY_SCOPE_AGENT 0
using std::min;
struct float4 { float x, y, z, w; };
struct double4 { double x, y, z, w; };
inline uint32_t atomicMin(uint32_t* p, uint32_t v) { const uint32_t o = *p; if (v < o) *p = v; return o; }
inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p = o + v; return o; }
inline uint32_t __hip_atomic_load(uint32_t* p, int, int) { return *p; }
inline void __hip_atomic_store(uint32_t* p, uint32_t v, int, int) { *p = v; }
inline bool __hip_atomic_compare_exchange_strong(uint32_t* p, uint32_t* expected, uint32_t desired, int, int, int) {
    if (*p == *expected) { *p = desired; return true; }
    *expected = *p;
    return false;
}
namespace msceer {
struct VGrid {
    int X, Y, Z;
    int64_t sxy;
    int64_t verts() const { return sxy * Z; }
};
}  // namespace msceer

#include "lines_core.hpp"

using namespace msceer;

// stats (8): saddles, windows, windows cut short by the pool, lines traced
//            alone, streamlines recorded, rounds, tape entries, entries linked
//            to an earlier list entry of their cell
extern "C" int emul_tapes(const float* f, long long X, long long Y, long long Z, const uint8_t* grad,
                          const double* field3, int8_t* restr, int asc, float ethr, float gthr, int iters,
                          long long window, long long chunks, long long* stats) {
    const CellGeom m{2 * X - 1, 2 * Y - 1, 2 * Z - 1, (2 * X - 1) * (2 * Y - 1)};
    const uint64_t C = (uint64_t)m.sxy * (uint64_t)m.Mz;
    const VGrid g{(int)X, (int)Y, (int)Z, X * Y};
    std::vector<double4> gd((size_t)(X * Y * Z));
    for (size_t v = 0; v < gd.size(); v++) gd[v] = double4{field3[3 * v], field3[3 * v + 1], field3[3 * v + 2], 0.0};
    const GradSrc<double> src{gd.data()};
    std::vector<uint64_t> keys;
    for (uint64_t c = 0; c < C; c++) {
        if (!critical(grad, (uint32_t)c)) continue;
        int64_t x, y, z;
        m.xyz((uint32_t)c, x, y, z);
        if ((int)((x & 1) + (y & 1) + (z & 1)) != (asc ? 2 : 1)) continue;
        int64_t best = -1;
        for (int k = 0; k < 8; k++) {
            if (((k & 1) && !(x & 1)) || ((k & 2) && !(y & 1)) || ((k & 4) && !(z & 1))) continue;
            const int64_t v = ((x >> 1) + (k & 1)) + X * (((y >> 1) + ((k >> 1) & 1)) + Y * ((z >> 1) + (k >> 2)));
            if (best < 0 || f[v] > f[best] || (!(f[best] > f[v]) && v > best)) best = v;
        }
        const float val = f[best];
        keys.push_back(((uint64_t)value_key(asc ? val : -1.0f * val) << 32) | c);
    }
    std::sort(keys.rbegin(), keys.rend());
    const uint64_t S = keys.size(), nslots = 7 * S;
    std::vector<uint32_t> slots(nslots);
    for (uint64_t k = 0; k < S; k++) saddle_seeds(grad, m, (uint32_t)keys[k], asc != 0, slots.data() + 7 * k);

    std::vector<uint64_t> pool((size_t)chunks * kTapeChunk), wmask((size_t)chunks);
    std::vector<uint32_t> stamp[2] = {std::vector<uint32_t>(C, kNoLine), std::vector<uint32_t>(C, kNoLine)};
    const int8_t target = asc ? 4 : 5;
    long long st[8] = {(long long)S, 0, 0, 0, 0, 0, 0, 0};
    uint64_t w0 = 0;
    while (w0 < nslots) {
        const uint32_t a0 = (uint32_t)w0, w1 = (uint32_t)std::min<uint64_t>(nslots, w0 + std::max<long long>(1, window));
        st[1]++;
        std::vector<uint32_t> head(w1 - a0, kNoLine), stop(w1 - a0, 0);
        uint32_t top = 0, wc = w1;
        for (uint32_t i = a0; i < w1; i++) {
            if (slots[i] == kNoLine || i % 7 == 6) continue;
            uint32_t hist[kHistory], vox = 0;
            TapeLabels lab{restr, target, a0 > 0, TapePool{pool.data(), (uint32_t)chunks, &top}, hist, 1u};
            trace_line(src, g, m, slots[i], asc != 0, (double)gthr, (double)ethr, iters, lab, &vox);
            lab.finish();
            st[4]++;
            if (lab.over) {
                wc = i;
                break;
            }
            head[i - a0] = lab.head;
            std::unordered_map<uint32_t, uint32_t> seen;
            for (uint32_t ch = lab.head; ch != kNoLine; ch = (uint32_t)pool[(size_t)ch * kTapeChunk]) {
                const uint32_t n = (uint32_t)(pool[(size_t)ch * kTapeChunk] >> 32);
                for (uint32_t k = 1; k <= n; k++) {
                    uint64_t& e = pool[(size_t)ch * kTapeChunk + k];
                    const uint32_t hi = (uint32_t)(e >> 32), c = (uint32_t)e, kind = (hi >> kKindShift) & 3u;
                    st[6]++;
                    const auto it = seen.find(c);
                    if (it != seen.end()) {
                        e = (uint64_t)((hi & ~kNoPrev) | it->second) << 32 | c;
                        st[7]++;
                    }
                    if (kind == kList) seen[c] = ch * kTapeChunk + k;
                }
            }
        }
        if (wc == a0) {
            // the first line's tape does not fit: it alone, in order
            DirectLabels lab{restr, target};
            uint32_t vox = 0;
            trace_line(src, g, m, slots[a0], asc != 0, (double)gthr, (double)ethr, iters, lab, &vox);
            st[3]++;
            w0 = a0 + 1;
            continue;
        }
        if (wc < w1) st[2]++;
        for (int round = 0;; round++) {
            st[5]++;
            bool changed = round == 0;
            std::vector<uint32_t>& in = stamp[round & 1];
            std::vector<uint32_t>& out = stamp[(round & 1) ^ 1];
            std::fill(out.begin(), out.end(), kNoLine);
            for (uint32_t i = a0; i < wc; i++) {
                if (slots[i] == kNoLine) continue;
                if (i % 7 == 6) {
                    out[slots[i]] = std::min(out[slots[i]], i);
                    continue;
                }
                TapeState s;
                uint32_t ended = 0, ord = 0;
                for (uint32_t ch = head[i - a0]; ch != kNoLine && !ended; ch = (uint32_t)pool[(size_t)ch * kTapeChunk]) {
                    const uint64_t* e = &pool[(size_t)ch * kTapeChunk];
                    const uint32_t n = (uint32_t)(e[0] >> 32);
                    uint64_t test = 0, exitm = 0, stopm = 0, first = 0, labm = 0, prevm = 0;
                    for (uint32_t k = 1; k <= n; k++) {
                        const uint64_t bit = 1ull << k;
                        const uint32_t hi = (uint32_t)(e[k] >> 32), c = (uint32_t)e[k], kind = (hi >> kKindShift) & 3u;
                        if (kind <= kExit) test |= bit;
                        if (kind == kExit) exitm |= bit;
                        if (kind == kStop) stopm |= bit;
                        if (hi & kFirst) first |= bit;
                        if (restr[c] == target || in[c] < i) labm |= bit;
                        if ((hi & kNoPrev) != kNoPrev) prevm |= bit;
                    }
                    auto own = [&](uint32_t k, uint64_t w) {
                        const uint32_t p = (uint32_t)(e[k] >> 32) & kNoPrev;
                        const uint64_t word = p / kTapeChunk == ch ? w : wmask[p / kTapeChunk];
                        return ((word >> (p % kTapeChunk)) & 1ull) != 0;
                    };
                    uint32_t at = 0;
                    const uint64_t w = tape_chunk(s, n, test, exitm, stopm, first, labm, prevm, own, &at);
                    if (round == 0 || wmask[ch] != w) changed = true;
                    wmask[ch] = w;
                    for (uint32_t k = 1; k <= n; k++)
                        if ((w >> k) & 1ull) out[(uint32_t)e[k]] = std::min(out[(uint32_t)e[k]], i);
                    if (at) ended = ord * kTapeChunk + at;
                    ord++;
                }
                if (stop[i - a0] != ended) changed = true;
                stop[i - a0] = ended;
            }
            if (!changed) break;
        }
        const std::vector<uint32_t>& fin = stamp[0];  // equal to stamp[1] now
        for (uint64_t c = 0; c < C; c++)
            if (fin[c] != kNoLine) restr[c] = target;
        std::fill(stamp[0].begin(), stamp[0].end(), kNoLine);
        std::fill(stamp[1].begin(), stamp[1].end(), kNoLine);
        w0 = wc;
    }
    if (stats) std::copy(st, st + 8, stats);
    return 0;
}
