// The times by which the prefill's plan (pd_python.cpp, on the host before the call) and its launches (pd_prefill.hip)
// choose among the kernels, in one place so that what is planned is what runs. Plain C++.
#pragma once

#include <stdint.h>

namespace pd {

// us per 32-key tile of a workgroup, one per CU, measured on MI355X (24 q / 4 kv heads): 192 rows, 256 rows, and a unit of
// the dealt launch's line (192 rows, K and V widened exactly, the planning and the seams of the pieces in it).
struct FaTimes {
    double tile, wide_tile, deal_unit;
};
constexpr FaTimes kFaTimes = {1.62, 1.85, 1.75};
constexpr FaTimes kFaTimesExact = {1.9, 2.2, 2.08};  // P' as fp16 hi + lo
constexpr const FaTimes& fa_times(bool exact) { return exact ? kFaTimesExact : kFaTimes; }

// Whether 256-row workgroups take less time for all rounds of one workgroup per CU: they have to save a round (2,048
// tokens x 4 splits: 3 rounds of 256 against 4, 2.92 ms against 3.30; 2,048 unsplit: one round of either, 3.7
// against 3.15).
constexpr bool fa_wide_saves(int64_t wide_rounds, int64_t rounds, bool exact) {
    return (double)wide_rounds * fa_times(exact).wide_tile < (double)rounds * fa_times(exact).tile;
}

// The deal of pd_prefill_balanced_kernel.
constexpr unsigned kFaSegmentUnits = 10;  // set-up and stores of a segment, ~16 us, in key tiles
constexpr unsigned kFaMinShare = 16;      // units of a workgroup: below, pieces cost more than they save
// An item is cut evenly where that gives no workgroup more than a share and this part of one.
constexpr unsigned kFaAlignedPart = 32;
// What the plan adds to an equal share: up to 20 more units in the longest workgroup (a share's ends fall on items'
// starts, and its last segment's set-up is its own), and planning on the device and merge, us. A dealt launch has to
// be rated 5 % faster.
constexpr int64_t kFaDealSpareUnits = 20;
constexpr double kFaDealFixedUs = 20.0;
constexpr double kFaDealMargin = 0.95;

}  // namespace pd
