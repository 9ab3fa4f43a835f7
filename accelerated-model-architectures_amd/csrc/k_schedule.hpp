// Order of the LDS reads, LDS-DMA loads, waits and barriers in the K loop of the persistent grouped GEMM kernel ("K loop by
// quadrants" in grouped_gemm.hip).  The kernel takes its loads and waits from here, and tests/k_schedule_check.cpp walks the
// same functions on the host: every half of an operand tile needs a barrier between its last read by any wave and the next
// load into its place, and a wait and a barrier between a load and the first read of what it brings.
#pragma once

namespace xma_rocm {
namespace k_schedule {

enum Half { Q0, Q1, P0, P1 }; // pieces 4 h .. 4 h + 3 of a K step's 16 LDS-DMA loads fill half h of the operand tiles

enum Mode {
    STEADY,        // step of a tile that overlaps: the loads of step kt + 2 go out in its slots (complete steps)
    OVL_FIRST,     // the same, first step: the second half of step 1's loads as well, and the row loads of the next tile
    OVL_SECOND,    // the same, the step behind that one: the waits leave the row loads in flight, too
    OVL_DRAIN,     // second-last step of such a tile: nothing is loaded
    OVL_LAST,      // its last step (stage 1; stage 0 is free): the next tile's first K step; no fragments are read ahead
    CHECKED,       // any step of any other tile (every piece checks that it lies inside K)
    CHECKED_FIRST, // the first of them
};

constexpr int ROW_LOADS = 5; // loads of row indices and scales per tile

// n-th piece in the order in which the halves are needed: Q0, P0, P1, Q1
constexpr int ordered(int n) { return n < 4 ? n : n < 12 ? n + 4 : n - 8; }

// What a slot loads: piece (-1: nothing) of the K step `ahead` steps after the current one (NEXT_TILE: step 0 of the next tile).
constexpr int NEXT_TILE = -1;
struct Load {
    int piece, ahead;
};
constexpr Load load_of(int mode, int phase, int slot) {
    if ((mode == OVL_FIRST || mode == CHECKED_FIRST) && phase < 2)
        return phase == 0 ? Load{ordered(8 + slot), 1} : Load{ordered(slot), 2};
    if (mode == OVL_LAST) return phase == 1 ? Load{8 + slot, NEXT_TILE} : phase == 2 ? Load{slot, NEXT_TILE} : Load{-1, 0};
    if (mode == OVL_DRAIN || (slot & 1) == 0) return Load{-1, 0};
    return Load{ordered(phase * 4 + slot / 2), 2};
}
// in front of the loop, between the MFMAs that produce the accumulators
constexpr Load load_before_loop(int slot) { return slot < 8 ? Load{ordered(slot), 1} : Load{-1, 0}; }
// row load of a slot, -1: none
constexpr int row_load_of(int mode, int phase, int slot) { return mode == OVL_FIRST && phase == 3 && slot >= 3 ? slot - 3 : -1; }

// The half that a phase reads from LDS, of the current step in phases 0 and 1, of the next one in phases 2 and 3.
constexpr Half read_of(int phase) { return phase == 0 ? P1 : phase == 1 ? Q1 : phase == 2 ? Q0 : P0; }
constexpr bool reads_ahead(int mode) { return mode != OVL_LAST; }

// Loads that the waits in front of the barriers leave in flight; -1: no wait for loads.  B stands between phases 1 and 2,
// A at the end of the step (not in OVL_LAST).
constexpr int in_flight_b(int mode) { return mode == OVL_LAST ? -1 : mode == OVL_DRAIN ? 8 : mode == OVL_SECOND ? 16 + ROW_LOADS : 16; }
constexpr int in_flight_a(int mode) { return mode == OVL_DRAIN ? 0 : mode == OVL_FIRST ? 16 + ROW_LOADS : 16; }

// Step 0's Q0 and P0 are read in front of the loop, and phase 1 of step 0 loads step 2 into their place: no barrier of the
// loop stands between the two.
constexpr bool BARRIER_BEFORE_LOOP = true;

} // namespace k_schedule
} // namespace xma_rocm
