// Every order in which the rhs, compute and store waves of a sweep can run, over the counters and rings of
// nlf_sweep_flow.hpp: a wave never reads a slot that holds another step's entry, and every run ends with all
// steps stored.  The external values' wave is taken to be done (it only delays the compute wave, which the orders
// cover).  The counters only grow and each rule only opens with them, so a wave that acts on older counters acts
// as it would now: a rule may be tested and acted on at one time.
//
// And the bound of a wait for another chunk: never shorter than all steps of the plan one after the other.
#include <array>
#include <cstdio>
#include <vector>

#include "nlf_sweep_flow.hpp"

using namespace nlf;

namespace {

constexpr int STEPS = 176, BLOCKS = STEPS / SWEEP_RB, BATCH = 8;   // BATCH: steps the store wave takes at a time

struct State {
    int block = 0, rhs = 0;              // rhs wave: block; 0 waits, 1 right-hand sides written, 2 first records written
    int computed = 0, compute = 0;       // compute wave: steps published; 0 waits, 1 read, 2 written
    int stored = 0, store = 0, m = 0;    // store wave: steps published; 0 waits, 1 took m steps, 2 read their first
                                         // records, 3 read their values
    size_t index() const {
        size_t i = size_t(block);
        i = i * 3 + size_t(rhs);
        i = i * (STEPS + 1) + size_t(computed);
        i = i * 3 + size_t(compute);
        i = i * (SWEEP_K + 1) + size_t(computed - stored);
        i = i * 4 + size_t(store);
        return i * (BATCH + 1) + size_t(m);
    }
};

// The ring slot of entry e holds it: it has been written, and the last entry written is less than a round ahead.
bool holds(int e, int last, int ring) { return e <= last && last - e < ring; }

}  // namespace

int main() {
    constexpr double READ = 0.2, STEP = 3.0, MARGIN = 4.0;     // us: the shortest read, the longest step
    for (long long steps = 1; steps <= (1ll << 31); steps *= 2)
        if (double(sweep_wait_reads(steps)) * READ < MARGIN * STEP * double(steps)) {
            std::printf("a wait ends before %lld steps\n", steps);
            return 1;
        }
    std::vector<bool> seen(size_t(BLOCKS + 1) * 3 * (STEPS + 1) * 3 * (SWEEP_K + 1) * 4 * (BATCH + 1));
    std::vector<State> todo{State{}};
    seen[State{}.index()] = true;
    size_t states = 0;
    while (!todo.empty()) {
        const State s = todo.back();
        todo.pop_back();
        ++states;
        bool moved = false;
        auto go = [&](const State& t) {
            moved = true;
            if (seen[t.index()]) return;
            seen[t.index()] = true;
            todo.push_back(t);
        };
        auto wrong = [&](const char* what, int e) {
            std::printf("%s of step %d is not in its slot: staging from %d (%d), computed %d, stored %d\n", what, e,
                        s.block * SWEEP_RB, s.rhs, s.computed, s.stored);
            return 1;
        };
        const int s0 = s.block * SWEEP_RB, staged = s0;
        const int last_rhs = s0 + (s.rhs >= 1 ? SWEEP_RB : 0) - 1;             // last right-hand side written
        const int last_first = s0 + (s.rhs >= 2 ? SWEEP_RB : 0);               // last first record written
        const int last_win = s.computed + (s.compute == 2 ? 1 : 0) - 1;        // last step in the window
        State t = s;
        if (s.block < BLOCKS) {
            if (s.rhs == 0 && sweep_rhs_free(s0, s.computed, s.stored)) { t.rhs = 1; go(t); }
            if (s.rhs == 1) { t.rhs = 2; go(t); }
            if (s.rhs == 2) { t.rhs = 0; ++t.block; go(t); }
        }
        t = s;
        if (s.compute == 0 && s.computed < staged && s.computed < sweep_window_end(s.stored)) {
            if (!holds(s.computed, last_rhs, SWEEP_R)) return wrong("the right-hand side", s.computed);
            t.compute = 1;
            go(t);
        }
        if (s.compute == 1) { t.compute = 2; go(t); }
        if (s.compute == 2) { t.compute = 0; ++t.computed; go(t); }
        t = s;
        if (s.store == 0)
            for (int m = 1; m <= BATCH && m <= s.computed - s.stored; ++m) { t.store = 1; t.m = m; go(t); }
        if (s.store == 1) {
            for (int k = 0; k <= s.m; ++k)
                if (!holds(s.stored + k, last_first, SWEEP_FIRST)) return wrong("the first record", s.stored + k);
            t.store = 2;
            go(t);
        }
        if (s.store == 2) {
            for (int k = 0; k < s.m; ++k)
                if (!holds(s.stored + k, last_win, SWEEP_K)) return wrong("the value", s.stored + k);
            t.store = 3;
            go(t);
        }
        if (s.store == 3) { t.store = 0; t.stored += s.m; t.m = 0; go(t); }
        if (!moved && s.stored != STEPS) {
            std::printf("stuck: staging from %d, computed %d, stored %d\n", s0, s.computed, s.stored);
            return 1;
        }
    }
    std::printf("%zu states\n", states);
    return 0;
}
