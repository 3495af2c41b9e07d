// Where a workgroup of the prefill attention kernel (fmha_fwd.hip) keeps the work items to come. Plain C++: the order of the accesses below is
// checked on the CPU.
#pragma once

namespace mi355 {

// Item `round` (1, 2, ..; item 0 is worked out by every wave for itself) is read by all waves during iteration `round` of the loop
// over the items and once more behind that iteration's last barrier, when it becomes the current one. Behind that same barrier the
// last wave may already be in the next iteration, where it writes the following kAtOnce items in front of the next barrier: so the
// entries form two halves that are written in turn, and what a slower wave still has to read is in the other one.
struct ListedItems {
    static constexpr int kAtOnce = 64;          // items written together, one per lane
    static constexpr int kHeld = 2 * kAtOnce;   // entries
    // whether items round .. round + kAtOnce - 1 are written at the start of iteration `round`
    static constexpr bool refill(int round) { return ((round - 1) & (kAtOnce - 1)) == 0; }
    static constexpr int entry(int round) { return (round - 1) & (kHeld - 1); }
};

}  // namespace mi355
