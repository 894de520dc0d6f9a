// When the waves of a triangular sweep (nlf_sweep.inl) may write to the rings in LDS that pass steps between
// them, and how long they wait for a value of another chunk.  Plain C++: the kernels ask these functions, and a test
// on the host walks every order in which the waves can run against them.
#pragma once

namespace nlf {

constexpr int SWEEP_K = 48;              // steps the LDS window holds
constexpr int SWEEP_R = 48;              // steps the right-hand side ring holds
constexpr int SWEEP_RB = 16;             // steps the rhs wave stages at a time
constexpr int SWEEP_FIRST = 2 * SWEEP_R; // entries of the ring of the steps' first records

// Steps the window has room for, by what the store wave has copied out.
constexpr int sweep_window_end(int stored) { return stored + SWEEP_K; }

// Whether the rhs wave may stage steps s0 .. s0 + SWEEP_RB - 1.  It overwrites the right-hand sides of the
// SWEEP_R steps before, which must be computed, and SWEEP_RB + 1 first records, s0 .. s0 + SWEEP_RB (a step's end
// is the next one's first record): the oldest, of step s0 + SWEEP_RB - SWEEP_FIRST, must not be wanted any more,
// and the store wave reads that of step `stored` next.
constexpr bool sweep_rhs_free(int s0, int computed, int stored) {
    return computed >= s0 + SWEEP_RB - SWEEP_R && stored > s0 + SWEEP_RB - SWEEP_FIRST;
}

// Reads of a missing value before it is taken as not-a-number: the end of a wait that no fault-free run reaches.  A
// chunk may wait for every step of the plan, which can follow each other one by one (a strip numbered along its short
// side: 8 million rows to a chunk, each a step of the factorisation).  64 reads per step are 12 us and more (a read is
// a round trip to the L2, 0.2 us at least); a step takes 0.1 to 0.2 us in a sweep and 1.6 to 3 us in the factorisation.
constexpr long long sweep_wait_reads(long long steps) { return (1ll << 21) + 64 * steps; }

}  // namespace nlf
