// When the waves of a triangular sweep (nlf_sweep.inl) may write to the rings in LDS that pass steps between
// them.  Plain C++: the kernel asks these functions, and a test on the host walks every order in which the waves
// can run against them.
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

}  // namespace nlf
