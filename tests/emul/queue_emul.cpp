// Host run of the re-integration queue's counting (test infrastructure):
// work_queue.hpp, the code the gfx950 kernel runs, by two participants whose
// atomic operations are interleaved in every possible way -- one does work (a
// chain through the queue, or through a trace ahead that is wanted), the other
// asks queue_drained() as a wave left with traces ahead does.  An answer of
// "drained" while work is still to be done is counted as wrong.
#include <ucontext.h>

#include <cstdint>
#include <functional>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_AGENT 0

namespace {

// A participant's code, run up to its next atomic operation at a time.
struct Party {
    ucontext_t self, back;
    std::vector<char> stack = std::vector<char>(1 << 16);
    std::function<void()> code;
    bool ended = false;
};
Party* g_now = nullptr;

void entry() {
    g_now->code();
    g_now->ended = true;
    swapcontext(&g_now->self, &g_now->back);
}
void begin(Party& p, std::function<void()> code) {
    p.code = std::move(code);
    getcontext(&p.self);
    p.self.uc_stack.ss_sp = p.stack.data();
    p.self.uc_stack.ss_size = p.stack.size();
    p.self.uc_link = nullptr;
    makecontext(&p.self, entry, 0);
}
void step(Party& p) {
    g_now = &p;
    swapcontext(&p.back, &p.self);
}
// before every atomic operation: the other one's turn
void turn() { swapcontext(&g_now->self, &g_now->back); }

}  // namespace

inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { turn(); const uint32_t o = *p; *p = o + v; return o; }
inline uint32_t __hip_atomic_load(const uint32_t* p, int, int) { turn(); return *p; }
inline bool __hip_atomic_compare_exchange_strong(uint32_t* p, uint32_t* expected, uint32_t desired, int, int, int) {
    turn();
    if (*p == *expected) { *p = desired; return true; }
    *expected = *p;
    return false;
}

#include "work_queue.hpp"

using namespace msceer;

namespace {

struct World {
    uint32_t head = 0, tail = 0, chunk_head = 0, first = 0, busy = 0;
    WorkQueue q{};
    bool finished = false;  // the worker has nothing left and can get nothing more
    World() {
        q.capacity = 1u << 20;
        q.head = &head;
        q.tail = &tail;
        q.chunk_head = &chunk_head;
        q.busy = &busy;
    }
};

void leave(World& w, bool& counted) {
    if (counted) atomicAdd(w.q.busy, 0xFFFFFFFFu);
    counted = false;
}

// 0: items through the queue, each queueing the next but the last
void through_queue(World& w) {
    bool counted = false;
    for (int left = 3; left > 0; left--) {
        uint32_t base = 0;
        if (queue_claim(w.q, 64, counted, &base) != 1) return;
        if (left > 1) atomicAdd(w.q.tail, 1u);
        if (left == 1) w.finished = true;
        leave(w, counted);
    }
}
// 1: an item reaches a vertex traced ahead; the wave that traces it, which
// holds nothing else, finishes it and queues one more
void through_trace(World& w) {
    bool counted = false, other = false;
    uint32_t base = 0;
    if (queue_claim(w.q, 64, counted, &base) != 1) return;
    atomicAdd(w.q.busy, 1u);  // wanted
    leave(w, counted);
    queue_takeover(w.q, 1, other);
    atomicAdd(w.q.tail, 1u);
    leave(w, other);
    if (queue_claim(w.q, 64, other, &base) != 1) return;
    w.finished = true;
    leave(w, other);
}
// 2: the last chunk of the pass-2 items, which queues one more
void through_chunk(World& w) {
    bool counted = false;
    uint32_t base = 0;
    queue_enter(w.q);
    counted = true;
    if (atomicAdd(w.q.chunk_head, 64u) >= w.first) return;
    atomicAdd(w.q.tail, 1u);
    leave(w, counted);
    if (queue_claim(w.q, 64, counted, &base) != 1) return;
    w.finished = true;
    leave(w, counted);
}

}  // namespace

// Wrong answers over all interleavings of scenario `kind`; runs[0]: how many
// interleavings, runs[1]: in how many the queue was found drained.
extern "C" long long emul_queue(int kind, long long* runs) {
    runs[0] = runs[1] = 0;
    long long wrong = 0;
    std::vector<int> plan;  // whose turn: 0 the worker, 1 the one who asks; the rest 0
    while (true) {
        World w;
        if (kind == 2) w.first = 64;
        else w.tail = 1;
        bool drained = false;
        Party worker, asker;
        begin(worker, [&] {
            if (kind == 0) through_queue(w);
            else if (kind == 1) through_trace(w);
            else through_chunk(w);
        });
        begin(asker, [&] {
            if (kind == 2) {
                // it asks only once no chunk is left for it
                queue_enter(w.q);
                const bool mine = atomicAdd(w.q.chunk_head, 64u) < w.first;
                bool counted = true;
                leave(w, counted);
                if (mine) return;
            }
            drained = queue_drained(w.q);
            if (drained && !w.finished) wrong++;
        });
        size_t at = 0;
        while (!asker.ended) {
            if (at == plan.size()) plan.push_back(worker.ended ? 1 : 0);
            if (plan[at] == 0 && worker.ended) plan[at] = 1;
            step(plan[at] ? asker : worker);
            at++;
        }
        plan.resize(at);
        runs[0]++;
        runs[1] += drained ? 1 : 0;
        // the next plan: the last worker's turn becomes the asker's
        while (!plan.empty() && plan.back() == 1) plan.pop_back();
        if (plan.empty()) return wrong;
        plan.back() = 1;
    }
}
